"""Superblock sums, scales and minimums at the ends of their ranges: the matrix-core kernels publish what
the sweeps and the generic kernel (the CPU path's bits) publish for the same pairs."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev(array, device):
    return torch.from_numpy(np.ascontiguousarray(array)).to(device)


# both token blocks of a tile, one, a tile of one pair more than the few-pair kernels take, and a remainder of theirs
POPULATIONS = [64 + 40, 33, 17, 5]


@pytest.mark.parametrize("qtype", ["Q4_K", "Q2_K", "IQ2_XXS"])
@pytest.mark.parametrize("scales,magnitude", [("ordinary", 1.0), ("largest", 2.0 ** 80), ("subnormal", 2.0 ** -108)])
def test_scales_and_minimums_reach_as_far_as_floats(gpu, oracle, qtype, scales, magnitude):
    """Sub-block scales and minimums at their largest against rows whose codes all have the largest magnitude and one sign,
    (the largest sums there are), with block scales whose products are ordinary, huge or denormal."""
    from yvex_amd import kernels as K
    qt, hidden, intermediate = getattr(oracle, qtype), 256, 512
    # (IQ2_XXS: codebook entries, signs and group scales at once)
    block, heads, halves = {"Q4_K": (144, slice(4, 16), (0, 2)), "Q2_K": (84, slice(0, 16), (80, 82)),
                            "IQ2_XXS": (66, slice(2, 66), (0,))}[qtype]
    first = qt if qtype == "IQ2_XXS" else oracle.Q4_K
    experts, pairs = len(POPULATIONS), sum(POPULATIONS)
    g = oracle.Generator(45, f"limits.{qtype}")
    up = dev(g.weights(first, experts * intermediate, hidden), gpu)
    down = g.weights(qt, experts * hidden, intermediate)
    blocks = down.reshape(-1, block)
    blocks[::2, heads] = 255
    if scales != "ordinary":
        bits = (np.full(len(blocks), 0x7800) if scales == "largest" else 1 + np.arange(len(blocks)) * 7 % 1023).astype(np.uint16)
        for offset in halves:
            blocks[:, offset], blocks[:, offset + 1] = bits & 255, bits >> 8
    weights = K.expert_weights(up, up, dev(down, gpu), (first, first, qt), hidden, intermediate)
    status = K.new_status(gpu)
    selected = torch.repeat_interleave(torch.arange(experts), torch.tensor(POPULATIONS)).reshape(pairs, 1).to(gpu)
    wl = K.worklist_build(selected, experts, status)
    x = g.normal(pairs * intermediate).reshape(pairs, intermediate)
    x[::3], x[1::3] = 1.0, -1.0
    x = (x / np.abs(x).max(axis=1, keepdims=True) * magnitude).astype(np.float32)
    act = K.q8k_quantize(dev(x, gpu), status)
    out = [torch.full((pairs, hidden), float("nan"), device=gpu) for _ in range(2)]
    K.moe_down(weights, act, True, wl, pairs, experts, out[0], status)
    K.moe_down_rows(weights, act, wl, pairs, experts, out[1], status)
    assert int(status.item()) == 0 and bool(torch.isfinite(out[0]).all())
    assert torch.equal(out[0].view(torch.int32), out[1].view(torch.int32))


# the same for a plain projection: 16 x 16, 32 x 32 and 32 x 64 tiles, those that share a compute unit, tiles staged through
# LDS; ragged edges on both sides; more 32 x 64 tiles of long rows than compute units
@pytest.mark.parametrize("rows,width,inputs", [(50, 512, 20), (2060, 768, 71), (2078, 512, 100), (8200, 256, 41), (8180, 256, 230),
                                               (2060, 6144, 530), (4100, 11520, 140)])
@pytest.mark.parametrize("scales,magnitude", [("ordinary", 1.0), ("largest", 2.0 ** 80), ("subnormal", 2.0 ** -108)])
def test_q4k_projections_reach_as_far_as_floats(gpu, oracle, rows, width, inputs, scales, magnitude):
    """Against the kernel of a few input rows, which scales on the vector ALU, for every row of the batch, and the CPU path's
    bits of some."""
    from yvex_amd import kernels as K
    g, status = oracle.Generator(48, f"q4k.limits.{rows}.{inputs}"), K.new_status(gpu)
    packed = g.weights(oracle.Q4_K, rows, width)
    blocks = packed.reshape(-1, 144)
    blocks[::2, 4:16] = 255
    if scales != "ordinary":
        bits = (np.full(len(blocks), 0x7800) if scales == "largest" else 1 + np.arange(len(blocks)) * 7 % 1023).astype(np.uint16)
        for offset in (0, 2):
            blocks[:, offset], blocks[:, offset + 1] = bits & 255, bits >> 8
    x = g.normal(inputs * width).reshape(inputs, width)
    x[::3], x[1::3] = 1.0, -1.0
    x = (x / np.abs(x).max(axis=1, keepdims=True) * magnitude).astype(np.float32)
    weights, rows_in = dev(packed, gpu), dev(x, gpu)

    def product(first, count):
        act = K.q8k_quantize(rows_in[first:first + count].contiguous(), status)
        return K.matvec(weights, oracle.Q4_K, rows, width, act, input_q8=True, input_rows=count, status=status)
    got = product(0, inputs)
    want = torch.cat([product(first, min(3, inputs - first)) for first in range(0, inputs, 3)])
    assert int(status.item()) == 0 and bool(torch.isfinite(got).all())
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    picked = [0, inputs // 2, inputs - 1]
    exact = oracle.q8_matvec(oracle.Q4_K, packed, rows, width, oracle.q8k_quantize(x[picked]), len(picked))
    assert np.array_equal(got[picked].cpu().numpy().view(np.uint32), exact.view(np.uint32))


# more 64-token tiles than compute units, a remainder of tokens and of rows, one superblock and fewer than a workgroup's waves
@pytest.mark.parametrize("rows,width,inputs", [(8200, 256, 70), (8224, 768, 97), (4112, 1536, 190)])
def test_q4k_tiles_that_share_a_compute_unit_publish_what_single_ones_do(gpu, oracle, rows, width, inputs):
    """The first 2048 rows alone are few enough tiles for a compute unit each; the order of every sum is the same."""
    from yvex_amd import kernels as K
    g, status = oracle.Generator(47, f"paired.{rows}.{width}"), K.new_status(gpu)
    weights = dev(g.weights(oracle.Q4_K, rows, width), gpu)
    act = K.q8k_quantize(dev(g.normal(inputs * width).reshape(inputs, width), gpu), status)
    units, few, tiles = torch.cuda.get_device_properties(gpu).multi_processor_count, 2048, (inputs + 63) // 64
    assert (rows + 31) // 32 * tiles > units >= few // 32 * tiles and (rows + 127) // 128 * tiles < units
    assert few // 16 * ((inputs + 31) // 32) > units            # (no 16 x 16 tiles)
    many, part = (K.matvec(weights[:count * width // 256 * 144], oracle.Q4_K, count, width, act, input_q8=True, input_rows=inputs,
                           status=status) for count in (rows, few))
    assert int(status.item()) == 0 and torch.equal(many[:, :few].contiguous().view(torch.int32), part.view(torch.int32))
