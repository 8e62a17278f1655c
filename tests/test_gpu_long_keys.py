"""Portions of prompts over one key of 256 or 512 elements for all heads, values of 64 or 128 apart from it, at the edges of the
kernel's tiles: 128 (query, head) rows a workgroup (short portions over up to 256 keys: 64 rows of a head), 64 keys a tile, two or one
key rows to a copy, pages that hold a tile and pages that do not, keys cut into slices in the single rows' room, and scores that meet a cap, a bias or both.  Bound: as the shorter keys'
portions have it (the products over 512 elements are fp32 sums of exact terms: 2^-24 sqrt(512) of their norm, below 2^-19)."""
import pytest

import test_gpu_row_attention as portions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,Dv,H,G,page,lens,ctxs,opts", [
    (512, 128, 28, 4, 64, [18, 2, 19], [0, 64, 700], dict(sink=True)),                           # 126, 14 and 133 rows
    (512, 128, 8, 4, 16, [70, 1, 33], [31, 0, 70], dict(window=90, keep=4)),                     # small pages
    (512, 64, 4, 2, 64, [129, 64], [1, 512], dict(window=70, keep=9, gate=True)),
    (256, 128, 6, 2, 128, [65, 3], [1000, 63], dict(chunk=300, elem=True)),
    (256, 64, 4, 4, 32, [64, 130], [64, 5], dict(window=200, keep=130)),
    (512, 128, 28, 4, 64, [9], [3000], dict(sink=True, gate=True)),                              # slices
    (512, 128, 28, 4, 64, [10, 10, 1], [1500, 2040, 900], dict(window=1024, keep=4)),            # with a single row among them
    (256, 64, 4, 2, 64, [5] + [1] * 40, [2500] + [31 * i for i in range(40)], dict(elem=True)),  # beside too many: whole
    (512, 128, 4, 2, 64, [1, 5, 1, 40, 1], [0, 3, 900, 100, 0], {}),                                # few keys: single rows among the blocks
    (512, 64, 4, 2, 64, [3, 70, 2], [-2, -30, -1], dict(sink=True)),                             # rows in front of their sequence
    (512, 128, 4, 2, 64, [70, 3], [200, 1000], dict(softcap=5.0)),
    (256, 128, 4, 2, 16, [70, 3], [200, 0], dict(bias="log", sink=True)),
    (512, 64, 4, 2, 64, [70, 3], [200, 1000], dict(softcap=5.0, bias="log", window=150, keep=3)),
    # few keys and few workgroups: up to 256 keys, up to 256 workgroups, single rows in the same launch or in the decode form's
    (512, 128, 28, 4, 64, [65, 17, 2], [191, 0, 63], dict(sink=True, gate=True)),                # 256 keys; a second block of one row
    (512, 128, 28, 4, 64, [65, 17, 2], [192, 0, 63], dict(sink=True, gate=True)),                # one more
    (256, 64, 4, 2, 16, [64, 1, 1], [100, 0, 255], dict(elem=True, bias="log")),                 # single rows along
    (512, 64, 4, 2, 32, [30] + [1] * 66, [100] + [3 * i for i in range(66)], dict(softcap=5.0)),  # too many: by the decode form
    (256, 128, 8, 4, 64, [33, 64] * 8, [5, 190] * 8, dict(sink=True)),                           # 128 workgroups
    (512, 64, 4, 2, 64, [65] * 40, [100] * 40, {}),                                              # 320
    (512, 128, 4, 2, 64, [70, 9], [300, 900], dict(window=100, keep=4)),                         # a window: few tiles of many
    (512, 64, 4, 2, 64, [63, 3], [-40, -2], dict(sink=True, chunk=50)),
    # few single rows beside cut keys: slices of 19 tiles, which their own launch takes, in front of whole and of cut portions; of 10, in
    # pages of a tile along with the portions, in smaller pages not
    (256, 64, 8, 2, 64, [700, 300, 1, 1], [0, 200, 2400, 1300], dict(sink=True)),
    (512, 128, 8, 2, 64, [700, 300, 1, 1], [1700, 2100, 2400, 1], dict(sink=True, gate=True)),
    (256, 128, 8, 2, 64, [339, 190, 1, 1], [0, 2500, 3000, 1300], {}),
    (256, 128, 8, 2, 16, [339, 190, 1, 1], [0, 2500, 3000, 1300], {}),
])
def test_portions_over_long_shared_keys(D, Dv, H, G, page, lens, ctxs, opts):
    portions.test_against_64_bits("shared", D, Dv, H, G, page, lens, ctxs, opts)
