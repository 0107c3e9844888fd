"""Figures that the benchmark derives, without a GPU."""
import bench


def test_policy_peak_prices_each_layer_at_its_instruction():
    """29-256-256-8: 7424 multiply-adds in f32, 67584 as six bf16 products; a
    net below 32 neurons runs in f32 throughout."""
    want = (7424 + 67584) / (7424 / 157.3 + 6 * 67584 / 2516.6)
    assert abs(bench.policy_peak_tflops(29, 256, 8) - want) < 1e-9 and 300 < want < 420
    assert abs(bench.policy_peak_tflops(29, 16, 8) - 157.3) < 1e-9
