"""bench.py's ceilings and FLOP counts (no GPU)."""
import bench


def test_path_flops_count_the_work_done():
    """Brute force over a settling's problems: with one-row layers, step t has the batch's size in layers up to t + 1."""
    for sizes, T in (([8192] * 12, 16), ([4096] * 6, 32), ([30, 20, 10, 5], 2), ([784, 256, 256, 10], 20), ([9, 4], 3)):
        B, L = 64, len(sizes)
        for shared in (False, True):
            want = 0
            for t in range(T):
                for l in range(1, L):
                    if not shared or l <= t + 1:
                        want += 2 * (2 * B * sizes[l] * sizes[l - 1])   # the error and the update problem
            assert bench.path_flops(sizes, B, T, shared) == want
    # 242 of 352 problems
    assert bench.path_flops([8192] * 12, 1, 16, True) / bench.path_flops([8192] * 12, 1, 16, False) == 242 / 352


def test_fp32_ceiling_follows_the_tile():
    c = bench.CONFIGS
    assert bench.mfma_peak(c["c1"]["sizes"], c["c1"]["batch"], "f32") == bench.PEAK["f32"]
    assert bench.mfma_peak(c["c2"]["sizes"], c["c2"]["batch"], "f32") == bench.PEAK["bf16"] / 6
    assert bench.mfma_peak(c["c2"]["sizes"], c["c2"]["batch"], "f32", 64) == bench.PEAK["f32"]
    assert bench.mfma_peak(c["c1"]["sizes"], c["c1"]["batch"], "f32", 128) == bench.PEAK["bf16"] / 6
    assert bench.mfma_peak(c["c5"]["sizes"], c["c5"]["batch"], "bf16") == bench.PEAK["bf16"]
