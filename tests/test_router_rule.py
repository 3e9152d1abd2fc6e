"""Which prompt-sized steps take their router's logits from the matrix cores (mixer_ops.router_tiles_win): only what the kernel takes, and nothing that the library
was measured to be faster at."""
import pytest

from gbx_lm_amd.mixer_ops import router_tiles_win


def test_only_what_the_kernel_takes():
    for t in (0, 1, 33, 511, 512, 700, 2048, 5000, 10 ** 6):
        for e in (0, 1, 5, 64, 128, 129, 256, 257, 4096):
            for k in (0, 4, 8, 100, 264, 1024, 1536, 2040, 2048, 2056, 7168):
                if router_tiles_win(t, e, k):
                    assert k % 8 == 0 and 0 < k <= 2048 and 0 < e <= 256 and e * k < 1 << 29 and 512 <= t and t * e <= 3 << 19


@pytest.mark.parametrize("t,e,k,tiles", [
    (512, 128, 1024, True), (512, 128, 1152, False), (512, 64, 2048, False), (1024, 64, 2048, False), (1024, 64, 1536, False), (1280, 64, 1536, True),
    (1536, 64, 2048, True), (3481, 128, 2048, True), (8192, 64, 2048, True), (2047, 256, 2048, True), (2500, 256, 2048, False), (8192, 256, 2048, False),
    (4500, 200, 1536, False), (2500, 256, 1024, True), (8192, 256, 1024, False), (12000, 128, 2048, True), (16000, 128, 2048, False)])
def test_sides_of_the_line(t, e, k, tiles):
    assert router_tiles_win(t, e, k) == tiles
