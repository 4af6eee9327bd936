"""Rule books by grids objects that are used again with fields of other sizes, on both sides of where a mask's ranks take
a scan over many workgroups (65536 words): the state of that scan is cleared by the kernel that writes or clears the mask,
and must not be taken for clear where it is another size's or has been used."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu

#            batch, field, window, pool, stride
SEQUENCE = [(3, 128, 3, 2, 2), (1, 9, 2, 2, 2), (3, 128, 3, 2, 2), (2, 131, 2, 2, 2), (9, 101, 3, 3, 2), (3, 128, 3, 2, 2),
            (1, 163, 3, 1, 1)]


def test_grids_used_again_with_other_sizes(scn, ctx):
    grids = [scn.Grids(ctx) for _ in range(3)]
    for turn, (batch, n, window, pool, stride) in enumerate(SEQUENCE):
        print("reuse", turn, batch, n, window, pool, flush=True)
        rng = np.random.default_rng(turn)
        per = 400
        key = np.concatenate([np.sort(rng.choice(n ** 3, per, replace=False)) for _ in range(batch)]).astype(np.int64)
        sample = np.repeat(np.arange(batch), per).astype(np.int32)
        row = (np.arange(batch * per) + sample + 1).astype(np.int32)
        bg = (np.arange(batch) * (per + 1)).astype(np.int32)
        ora = orc.Grids.from_flat(batch, sample, key, row, bg)
        grids[0].build(batch, 3, n, sample, key, row, bg, batch * (per + 1))
        n1 = n - window + 1
        n2 = (n1 - pool) // stride + 1
        for i, (a, b, size, step) in enumerate([(n, n1, window, 1), (n1, n2, pool, stride)]):
            ora, want, rows = orc.rules_square(ora, 3, a, b, size, step, 1)
            got = grids[i].plan_square(grids[i + 1], a, b, size, step)
            assert got == rows
            rules = ctx.empty(rows * size ** 3, np.int32)
            grids[i].fill(grids[i + 1], rules, rows * size ** 3)
            assert np.array_equal(rules.download(), want)
