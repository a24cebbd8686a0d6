"""The picked experts of a prompt's rows, in tiles of 128 pairs of one expert, against double precision."""
import pytest

from test_routed_experts_gpu import Experts, check

pytestmark = pytest.mark.gpu


# one line of K, outputs that end inside a tile of 64, 128 or 256 weight rows, experts without a pair and with less or more
# than a tile of them; widths that are no whole lines, which are staged through registers; enough tiles for the wide ones
# in the first product, in the second and in both
@pytest.mark.parametrize("E,D,F,rows,top", [(1, 64, 64, 256, 1), (3, 192, 320, 300, 2), (40, 320, 192, 700, 3), (2, 128, 1344, 129, 2),
                                            (4, 80, 48, 300, 2), (8, 256, 2112, 2000, 2), (8, 2112, 256, 2000, 2), (3, 1024, 1100 // 64 * 64, 5000, 3)])
def test_grouped_experts(E, D, F, rows, top):
    norm, worst = check(Experts(E, D, F), rows, top, adds=rows % 2 == 1)
    # the hidden units are rounded to eight bits (2^-9 each, and independent of each other)
    assert norm < 4e-3 and worst < 2e-2, (norm, worst)


def test_grouped_experts_identity_picks_clamps_and_weights_on_the_input():
    assert check(Experts(4, 128, 192, identity=3), 300, 5)[0] < 4e-3
    assert check(Experts(4, 128, 192, act=1, weight_on_input=1), 300, 3)[0] < 4e-3


def test_rows_of_a_prompt_need_not_begin_at_16_bytes():
    import torch
    x = Experts(4, 128, 192, identity=1)
    h = torch.randn(300, 128, generator=x.gen, device="cuda:0").bfloat16()
    ids, w, words = x.picks(300, 3)
    aligned = x.run(h, words, 3, torch.ones(300, 128, device="cuda:0"), True)
    room = torch.ones(300 * 128 + 1, device="cuda:0")
    assert torch.equal(x.run(h, words, 3, room[1:].view(300, 128), True), aligned) and float(room[0]) == 1.0
