"""f32 BGR rows of the input stage around the block width of 64 cells (NN2 works in 2x2 cells), in rows
cut out of wider ones so that their start is aligned or not, for every pattern.  Bit for bit against
the oracle, and nothing outside the rows is written."""
import numpy as np
import pytest

from oracle import debayer as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algo", [D.NN2, D.SP, D.MATRIX, D.NN, D.EA])
@pytest.mark.parametrize("h,w", [(2, 2), (2, 128), (14, 62), (8, 126), (10, 128), (6, 130), (18, 260)])
@pytest.mark.parametrize("colorid", [8, 9, 10, 11])
def test_every_row_store(algo, h, w, colorid):
    import torch

    import serstacker_amd as S

    n = 2
    raw = np.random.default_rng(w + algo).integers(0, 4096, (n, h, w)).astype(np.uint16)
    slab = torch.from_numpy(raw.view(np.int16)).cuda()
    want = [D.read_input_frame(raw[i], colorid, 12, algo, None, None) for i in range(n)]
    oh, ow = want[0].shape[:2]
    for off, pad in ((0, 0), (4, 8), (1, 3)):
        wide = torch.full((n, oh, ow + pad, 3), -1.0, dtype=torch.float32, device="cuda")
        outs = [wide[i, :, off:off + ow] for i in range(n)]
        S.read_input_frames([slab[i] for i in range(n)], colorid, 12, algo, outs=outs)
        got = wide.cpu().numpy()
        for i in range(n):
            np.testing.assert_array_equal(got[i, :, off:off + ow], want[i])
            assert (got[i, :, :off] == -1).all() and (got[i, :, off + ow:] == -1).all()
