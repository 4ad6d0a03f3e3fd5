"""How short traversal queues are dealt to the waves of a launch
(convector_amd/csrc/kernels.hip, deal_rays and Deal::position), enumerated on
the CPU: every queue position below n goes to exactly one wave, and none at or
above n, or a ray would be traversed twice, skipped, or read out of bounds --
for grids that are a multiple of the 8 XCDs, as all of a 256-CU device are, and
for others, which deal without regard to the XCD."""
import numpy as np
import pytest

DEAL_LANES, DEAL_SIMDS = 4, 1024


def _shares(n, grid, bw, whole_stripes):
    """Per wave of the launch (workgroup, wave): its queue positions."""
    waves = grid * bw
    whole = n // (64 * waves) * 64 if whole_stripes else 0
    left = n - whole * waves
    rest = -(-left // waves)
    blocks = grid
    if whole == 0:
        rest = max(rest, min(max(-(-n // DEAL_SIMDS), DEAL_LANES), 64))
        blocks = -(-n // (rest * bw))
    per_xcd = -(-blocks // 8)
    for block in range(grid):
        b = block
        if grid % 8 == 0:
            b = (b & 7) * per_xcd + (b >> 3) if (b >> 3) < per_xcd else blocks
        for wave in range(bw):
            mine = min(b, blocks) * bw + wave
            at = mine * rest if b < blocks else left
            end = (whole if b < blocks else 0) + (min(rest, left - at) if at < left else 0)
            l = np.arange(end, dtype=np.int64)
            if whole_stripes:
                yield np.where(l < whole, ((l >> 6) * waves + mine) * 64 + (l & 63),
                               whole * waves + mine * rest + (l - whole))
            else:
                yield mine * rest + l


@pytest.mark.parametrize("whole_stripes", [True, False])
@pytest.mark.parametrize("grid,bw", [(8, 1), (64, 4), (768, 1), (256, 2), (1, 1), (3, 4), (63, 1),
                                     (65, 2), (100, 4), (761, 1)])
def test_every_ray_is_dealt_once(grid, bw, whole_stripes):
    lanes = grid * bw * 64
    sizes = [1, 3, 4, 5, 63, 64, 65, 4096, 4097, lanes - 1, lanes]
    # hits-only queries of up to 8 rays per lane; records and bounces of up to one
    if whole_stripes:
        sizes += [lanes + 1, lanes + 4097, 4 * lanes - 63, 4 * lanes, 8 * lanes - 1, 8 * lanes]
    for n in sizes:
        if n > (8 if whole_stripes else 1) * lanes:
            continue
        seen = np.zeros(n, np.int64)
        for q in _shares(n, grid, bw, whole_stripes):
            assert len(q) == 0 or (q.min() >= 0 and q.max() < n), (n, grid, bw)
            seen[q] += 1
        assert (seen == 1).all(), (n, grid, bw)
