"""The launches around the projections: what an operation publishes to the host, and the small
kernels a layer's launch sequence is made of, at the edges of their ranges."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbytes", [0, 4, 1028, 65536])
def test_publish_brings_results_and_status_to_the_host(gpu, nbytes):
    from yvex_amd import load_library
    lib = load_library()
    host = C.c_void_p()
    assert lib.yvex_hip_host_alloc(C.byref(host), C.c_uint64(64 + 65536)) == 0
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    data = torch.arange(max(nbytes // 4, 1), dtype=torch.int32, device=gpu) * 3 + 1
    status = torch.tensor([2], dtype=torch.int32, device=gpu)
    seen = C.c_int(-1)

    def publish(count, clear, sequence):
        return lib.yvex_hip_publish(C.c_void_p(data.data_ptr()), C.c_uint64(count), C.c_void_p(status.data_ptr()),
                                    C.c_int(clear), host, C.c_uint32(sequence), stream)
    try:
        for sequence, clear, want in ((1, 0, 2), (2, 1, 2), (3, 1, 0)):      # kept, then cleared, then clear
            assert publish(nbytes, clear, sequence) == 0
            assert lib.yvex_hip_await(host, C.c_uint32(sequence), C.byref(seen), stream) == 0
            assert seen.value == want
            got = np.ctypeslib.as_array((C.c_int32 * (nbytes // 4)).from_address(host.value + 64))
            assert np.array_equal(got, data.cpu().numpy()[:nbytes // 4])
        assert publish(65540, 1, 4) == -7 and publish(2, 1, 4) == -10
    finally:
        torch.cuda.synchronize()
        lib.yvex_hip_host_free(host)


def ptr(t):
    return C.c_void_p(0 if t is None else t.data_ptr())


def u64(v):
    return C.c_uint64(v)


def call(name, *args):
    from yvex_amd import kernels as K
    K._call(name, *args, C.c_void_p(torch.cuda.current_stream().cuda_stream))


def dev(a, device):
    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def same_bits(a, b):
    return torch.equal(a.contiguous().view(torch.int32), b.contiguous().view(torch.int32))


# every kernel whose launch ends the operation by itself: the product that quantizes, the Q8_0 and IQ2_XXS 16 x 16 tiles, the
# Q4_K ones on eight and on four waves, a row and a few of superblock formats, the 256 x 32 tiles of an output head; one
# workgroup, fewer than counters, ragged numbers of them. `launches`: 1 where that is all, 2 with the quantizer's
@pytest.mark.parametrize("qtype,weight_rows,width,inputs,launches", [
    ("Q8_0", 1, 256, 1, 1), ("Q8_0", 4099, 512, 2, 1), ("Q8_0", 4096, 2304, 3, 2), ("Q8_0", 37, 256, 17, 2), ("Q8_0", 65281, 256, 3, 2),
    ("Q4_K", 250, 512, 19, 2), ("Q4_K", 8200, 256, 33, 3), ("Q4_K", 8200, 256, 31, 2), ("Q4_K", 9, 768, 1, 2), ("Q4_K", 1030, 512, 3, 2),
    ("IQ2_XXS", 52, 1024, 9, 2), ("IQ2_XXS", 300, 512, 1, 2), ("IQ2_XXS", 301, 1024, 4, 2), ("Q2_K", 70, 512, 2, 2)])
def test_projections_that_publish_for_themselves(gpu, oracle, qtype, weight_rows, width, inputs, launches):
    from backend_helpers import Backend
    from yvex_amd import abi, kernels as K
    qt, g, b = getattr(oracle, qtype), oracle.Generator(17, "publishing"), Backend()
    encoded = g.weights(qt, weight_rows, width)
    at = 80 if qtype == "Q2_K" else 0
    encoded[at:at + 2] = (0x53, 0x7b)           # a block scale of 60 000: rows of 3e38 overflow, in the product
    x = g.normal(inputs * width).reshape(inputs, width)
    try:
        _, base = b.resident(encoded)
        b.workspace(inputs * (width // 256) * 292 + 4096)
        out, facts, err = b.empty_f32(inputs * weight_rows), abi.OperationFacts(), abi.Error()
        good, huge = b.f32(x), b.f32(np.full_like(x, 3e38))

        def run(rows_in):
            return b.lib.yvex_rocm_encoded_matvec(b.handle, base, encoded.nbytes, qt, weight_rows, width, encoded.nbytes // weight_rows,
                                                  inputs, rows_in, None, 0, None, out, 1, C.byref(facts), C.byref(err))
        st = K.new_status(gpu)

        def product(rows_in):
            return K.matvec(dev(encoded, gpu), qt, weight_rows, width, K.q8k_quantize(dev(rows_in, gpu), st), input_q8=True,
                            input_rows=inputs, status=st).cpu().numpy()
        want = product(x)
        assert int(st.item()) == 0
        for _ in range(2):
            for _ in range(3):
                assert run(good) == 0, err.message
                assert facts.kernel_launches == launches
                got = b.read_f32(out, inputs * weight_rows).reshape(inputs, weight_rows)
                assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
            # what the product raises is this operation's, and the next one's word is clean
            assert run(huge) == abi.FORMAT
    finally:
        b.close()


# the most work that a launch ends by itself, and a little more: rows a wave of the product that quantizes, a
# compute unit for each IQ2_XXS tile and for five Q4_K ones, the longest rows that a wave has two of
@pytest.mark.parametrize("qtype,weight_rows,width,inputs,launches", [
    ("Q8_0", 32768, 256, 1, 1), ("Q8_0", 32769, 256, 1, 2), ("Q8_0", 32768, 512, 2, 1), ("Q8_0", 36001, 512, 2, 2),
    ("IQ2_XXS", 4096, 512, 16, 2), ("IQ2_XXS", 2048, 512, 17, 2), ("IQ2_XXS", 4100, 512, 7, 3), ("IQ2_XXS", 1376, 1024, 33, 3),
    ("Q4_K", 20480, 256, 13, 2), ("Q4_K", 20481, 256, 13, 3), ("Q4_K", 10250, 512, 32, 3),
    ("Q4_K", 24, 4096, 1, 2), ("Q4_K", 24, 4352, 1, 3), ("Q2_K", 24, 4096, 3, 2), ("Q2_K", 24, 4352, 3, 3), ("IQ2_XXS", 22, 4608, 2, 3)])
def test_where_projections_publish_for_themselves(gpu, oracle, qtype, weight_rows, width, inputs, launches):
    from backend_helpers import Backend
    from yvex_amd import abi, kernels as K
    assert torch.cuda.get_device_properties(gpu).multi_processor_count == 256
    qt, g, b, st = getattr(oracle, qtype), oracle.Generator(18, "published.lines"), Backend(), K.new_status(gpu)
    few = g.weights(qt, 64, width)
    encoded = np.tile(few, (weight_rows + 63) // 64)[:len(few) // 64 * weight_rows]
    x = g.normal(inputs * width).reshape(inputs, width)
    try:
        _, base = b.resident(encoded)
        b.workspace(inputs * (width // 256) * 292 + 4096)
        rows_in, out, facts, err = b.f32(x), b.empty_f32(inputs * weight_rows), abi.OperationFacts(), abi.Error()
        for _ in range(2):
            assert b.lib.yvex_rocm_encoded_matvec(b.handle, base, encoded.nbytes, qt, weight_rows, width, encoded.nbytes // weight_rows,
                                                  inputs, rows_in, None, 0, None, out, 1, C.byref(facts), C.byref(err)) == 0, err.message
            assert facts.kernel_launches == launches
        want = K.matvec(dev(encoded, gpu), qt, weight_rows, width, K.q8k_quantize(dev(x, gpu), st), input_q8=True, input_rows=inputs,
                        status=st).cpu().numpy()
        got = b.read_f32(out, inputs * weight_rows).reshape(inputs, weight_rows)
        assert int(st.item()) == 0 and np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        b.close()


# a full round of 128 x 128 tiles with ragged edges on both sides, one and three superblocks a row
@pytest.mark.parametrize("rows,width,inputs", [(2047, 256, 2040), (1921, 768, 2048)])
def test_q8_0_wide_tiles_are_the_oracles_bits(gpu, oracle, rows, width, inputs):
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"wide.{rows}.{width}.{inputs}")
    w, x = g.weights(oracle.Q8_0, rows, width), g.normal(inputs * width).reshape(inputs, width)
    status = K.new_status(gpu)
    act = K.q8k_quantize(dev(x, gpu), status)
    got = K.matvec(dev(w, gpu), oracle.Q8_0, rows, width, act, input_q8=True, input_rows=inputs, status=status).cpu().numpy()
    assert int(status.item()) == 0
    picked = np.array([0, 1, 31, 32, 63, 64, 127, 128, inputs // 2, inputs - 2, inputs - 1])
    encoded = oracle.q8k_quantize(x[picked])
    want = oracle.q8_matvec(oracle.Q8_0, w, rows, width, encoded, picked.size)
    assert np.array_equal(got[picked].view(np.uint32), want.view(np.uint32))


# a shape of each Q8_0 kernel: the lane chain, 16 x 16, 32 x 32, 256 x 32, 64 x 64, 128 x 64 and 128 x 128 tiles; 32 x 32 tiles
# that outnumber the compute units, long rows and not, and two rounds of 64 x 64 ones
@pytest.mark.parametrize("rows,width,inputs", [(33, 1024, 1), (100, 768, 20), (2047, 512, 95), (65300, 256, 9), (4090, 256, 200),
                                               (8190, 256, 230), (2047, 512, 2040),
                                               (2044, 7168, 321), (1022, 4096, 161), (7166, 2048, 130)])
@pytest.mark.parametrize("scales,magnitude", [("largest", 2.0 ** 95), ("subnormal", 2.0 ** -108)])
def test_q8_0_block_scales_reach_as_far_as_floats(gpu, oracle, rows, width, inputs, scales, magnitude):
    """Products of a weight and an input block's scale near either end of the float range, the sums of some
    blocks zero: the oracle's bits at every batch size."""
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"range.{scales}.{rows}.{width}.{inputs}")
    w = g.weights(oracle.Q8_0, rows, width)
    blocks = w.reshape(-1, 34)
    # (2^15, or the fp16 subnormals by turns)
    bits = np.full(len(blocks), 0x7800) if scales == "largest" else 1 + np.arange(len(blocks)) * 7 % 1023
    blocks[:, 0], blocks[:, 1] = bits & 255, bits >> 8
    blocks[::5, 2:] = 0
    x = g.normal(inputs * width).reshape(inputs, width)
    x = (x / np.abs(x).max() * magnitude).astype(np.float32)
    status = K.new_status(gpu)
    act = K.q8k_quantize(dev(x, gpu), status)
    got = K.matvec(dev(w, gpu), oracle.Q8_0, rows, width, act, input_q8=True, input_rows=inputs, status=status).cpu().numpy()
    assert int(status.item()) == 0
    picked = np.unique([0, inputs // 3, inputs // 2, max(inputs - 2, 0), inputs - 1])
    want = oracle.q8_matvec(oracle.Q8_0, w, rows, width, oracle.q8k_quantize(x[picked]), picked.size)
    assert np.all(np.isfinite(want)) and np.array_equal(got[picked].view(np.uint32), want.view(np.uint32))


# IQ2_XXS tiles whose waves share the row width: ragged on both sides, fewer superblocks than waves and a round of them and
# some, the last superblock of the matrix, either side of the line to the row-batch kernels
@pytest.mark.parametrize("rows,width,inputs", [(4, 512, 6), (20, 1024, 17), (132, 2560, 40), (500, 4608, 33), (1028, 8192, 16),
                                               (2048, 512, 96), (2048, 512, 97), (4100, 4096, 50)])
def test_iq2_tiles_of_small_matrices_are_the_oracles_bits(gpu, oracle, rows, width, inputs):
    from yvex_amd import kernels as K
    qt, g = oracle.IQ2_XXS, oracle.Generator(42, f"iq2.small.{rows}.{width}.{inputs}")
    w, x = g.weights(qt, rows, width), g.normal(inputs * width).reshape(inputs, width)
    status = K.new_status(gpu)
    act = K.q8k_quantize(dev(x, gpu), status)
    got = K.matvec(dev(w, gpu), qt, rows, width, act, input_q8=True, input_rows=inputs, status=status)
    rounded = K.matvec(dev(w, gpu), qt, rows, width, act, input_q8=True, input_rows=inputs, output_bf16=True, status=status)
    want = torch.from_numpy(oracle.q8_matvec(qt, w, rows, width, oracle.q8k_quantize(x), inputs)).to(gpu)
    assert same_bits(got, want) and same_bits(rounded, want.to(torch.bfloat16).float())
    assert int(status.item()) == 0


# one launch that quantizes its input rows: fewer rows than waves, rows whose blocks fill the lanes' chunks or not,
# rows on dword boundaries and between them, more weight rows than a round of waves
@pytest.mark.parametrize("rows,width,inputs,offset", [(1, 256, 1, 0), (17, 2048, 2, 2), (33, 2304, 1, 0), (100, 4096, 2, 0),
                                                      (130, 4352, 1, 2), (4099, 7168, 2, 0), (4100, 14336, 1, 2), (9000, 512, 2, 0)])
def test_quantizing_projection_is_quantization_and_projection(gpu, oracle, rows, width, inputs, offset):
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"quantizing.{rows}.{width}.{inputs}")
    held = torch.zeros(rows * width // 32 * 34 + offset, dtype=torch.uint8, device=gpu)
    held[offset:] = dev(g.weights(oracle.Q8_0, rows, width), gpu)
    w = held[offset:]
    x, add = (dev(g.normal(inputs * n).reshape(inputs, n), gpu) for n in (width, rows))
    status = K.new_status(gpu)
    lib, row_bytes = K.load_library(), width // 32 * 34
    assert lib.yvex_hip_matvec_quantizing_supported(ptr(w), C.c_uint(oracle.Q8_0), u64(rows), u64(width), u64(row_bytes), u64(inputs))

    def run(values, additive, bf16):
        out = torch.full((inputs, rows + 3), 7.0, device=gpu)
        call("yvex_hip_matvec_quantizing", ptr(w), C.c_uint(oracle.Q8_0), u64(rows), u64(width), u64(row_bytes), ptr(values),
             u64(inputs), u64(width), ptr(additive), ptr(out), u64(rows + 3), C.c_int(bf16), ptr(status))
        assert torch.all(out[:, rows:] == 7.0)
        return out[:, :rows]
    act = K.q8k_quantize(x, status)
    for additive, bf16 in ((None, 0), (add, 1)):
        padded = torch.zeros((inputs, rows + 3), device=gpu)
        if additive is not None:
            padded[:, :rows] = additive
        want = K.matvec(w, oracle.Q8_0, rows, width, act, input_q8=True, input_rows=inputs, status=status,
                        additive=additive, output_bf16=bool(bf16))
        assert same_bits(run(x, None if additive is None else padded, bf16), want)
    assert int(status.item()) == 0
    x[inputs - 1, width - 1] = float("nan")
    run(x, None, 0)
    assert int(status.item()) == 1
    # what it does not serve it refuses: three rows, rows on odd addresses, another format
    for at, qtype, n in ((w, oracle.Q8_0, 3), (held[offset + 1:], oracle.Q8_0, inputs), (w, oracle.Q4_K, inputs)):
        assert not lib.yvex_hip_matvec_quantizing_supported(ptr(at), C.c_uint(qtype), u64(rows), u64(width), u64(row_bytes), u64(n))


# 16 x 16 tiles on eight waves and on four, and the 32 x 32 and 16 x 16 Q8_0 tiles, the latter between 16-byte boundaries: ragged on both sides, fewer superblocks than
# waves, a superblock more than a round of them, one row against many
@pytest.mark.parametrize("qtype,rows,width,inputs", [
    ("Q4_K", 1, 256, 61), ("Q4_K", 17, 2304, 33), ("Q4_K", 4094, 1280, 19), ("Q4_K", 2065, 512, 31), ("Q4_K", 500, 2816, 66),
    ("Q8_0", 1, 256, 61), ("Q8_0", 17, 1280, 33), ("Q8_0", 2047, 1792, 95), ("Q8_0", 8201, 1024, 2),
    ("Q8_0", 1, 256, 12), ("Q8_0", 33, 2304, 16), ("Q8_0", 1001, 2816, 31), ("Q8_0", 4095, 512, 11)])
def test_dense_tiles_with_ragged_edges_are_the_oracles_bits(gpu, oracle, qtype, rows, width, inputs):
    from yvex_amd import kernels as K
    qt = getattr(oracle, qtype)
    g = oracle.Generator(42, f"ragged.{qtype}.{rows}.{width}.{inputs}")
    w, x = g.weights(qt, rows, width), g.normal(inputs * width).reshape(inputs, width)
    status = K.new_status(gpu)
    act = K.q8k_quantize(dev(x, gpu), status)
    held = torch.zeros(w.size + 4, dtype=torch.uint8, device=gpu)
    held[4:] = dev(w, gpu)
    for weights in (dev(w, gpu),) if qtype == "Q4_K" else (dev(w, gpu), held[4:]):
        got = K.matvec(weights, qt, rows, width, act, input_q8=True, input_rows=inputs, status=status).cpu().numpy()
        assert int(status.item()) == 0
        want = oracle.q8_matvec(qt, w, rows, width, oracle.q8k_quantize(x), inputs)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("rows,width,inputs", [(34, 512, 1), (128, 256, 5), (2048, 512, 17), (70, 768, 40)])
def test_q8_0_pair_is_two_projections(gpu, oracle, rows, width, inputs):
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"pair.{rows}.{width}.{inputs}")
    first, second = (dev(g.weights(oracle.Q8_0, rows, width), gpu) for _ in range(2))
    status = K.new_status(gpu)
    act = K.q8k_quantize(dev(g.normal(inputs * width).reshape(inputs, width), gpu), status)
    out = [torch.full((inputs, rows), 7.0, device=gpu) for _ in range(2)]
    call("yvex_hip_matvec_q8_0_pair", ptr(first), ptr(second), u64(rows), u64(width), u64(width // 32 * 34), ptr(act),
         u64(inputs), ptr(out[0]), ptr(out[1]), ptr(status))
    for w, got in zip((first, second), out):
        want = K.matvec(w, oracle.Q8_0, rows, width, act, input_q8=True, input_rows=inputs, status=status)
        assert same_bits(got, want)
    assert int(status.item()) == 0


@pytest.mark.parametrize("rows,experts,topk,width,bias", [(8, 8, 2, 1024, True), (33, 200, 16, 1024, False),
                                                          (255, 256, 8, 7168, True), (300, 24, 6, 2048, False)])
def test_router_joins_and_routes_in_one_launch(gpu, oracle, rows, experts, topk, width, bias):
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"routed.{rows}.{experts}")
    w = dev(g.normal(experts * width, width ** -0.5).reshape(experts, width), gpu)
    x = dev(g.normal(rows * width).reshape(rows, width), gpu)
    b = dev(g.normal(experts, 0.1).astype(np.float32), gpu) if bias else None
    status = K.new_status(gpu)
    logits = K.matvec_f32_rows(w, x, status)
    want = K.moe_route_rows(logits, b, topk, K.SIGMOID, True, 1.5, status)
    lib = K.load_library()
    lib.yvex_hip_matvec_f32_scratch_bytes.restype = C.c_uint64
    need = lib.yvex_hip_matvec_f32_scratch_bytes(u64(experts), u64(width), u64(rows))
    assert need > 0
    scratch = torch.empty(need, dtype=torch.uint8, device=gpu)
    got_logits = torch.empty_like(logits)
    selected, weights = torch.empty_like(want[0]), torch.empty_like(want[1])
    call("yvex_hip_matvec_f32_rows_routed", ptr(w), u64(experts), u64(width), ptr(x), u64(rows), u64(width), ptr(got_logits),
         ptr(b), u64(topk), C.c_int(K.SIGMOID), C.c_int(1), C.c_double(1.5), ptr(selected), ptr(weights), ptr(scratch),
         u64(need), ptr(status))
    assert same_bits(got_logits, logits) and torch.equal(selected, want[0]) and same_bits(weights, want[1])
    # ... and the preparation behind it: the worklist and the quantization alone
    wl, mine = K.worklist_build(selected, experts, status), K.Worklist(rows * topk, experts, gpu)
    encoded = torch.empty(rows * (width // 256) * 292, dtype=torch.uint8, device=gpu)
    call("yvex_hip_moe_prepare_routed", ptr(selected), u64(rows), u64(experts), u64(topk), *K._wl_ptrs(mine), ptr(x),
         u64(width), u64(width), ptr(encoded), ptr(status))
    for name in ("order", "expert_ids", "bucket_offsets", "bucket_populations", "sweep_offsets", "counts"):
        assert torch.equal(getattr(mine, name), getattr(wl, name)), name
    assert torch.equal(encoded, K.q8k_quantize(x, status)) and int(status.item()) == 0


@pytest.mark.parametrize("rows,shared,width", [(1, 1, 256), (7, 5, 768), (40, 3, 2048)])
def test_quantization_forms_the_shared_experts_products(gpu, oracle, rows, shared, width):
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"qswiglu.{rows}.{width}")
    values = dev(g.normal(rows * width).reshape(rows, width), gpu)
    gate, up = (dev(g.normal(shared * width, 4.0).reshape(shared, width), gpu) for _ in range(2))
    status = K.new_status(gpu)
    products = torch.empty_like(gate)
    call("yvex_hip_moe_swiglu_rows", ptr(gate), ptr(up), u64(shared * width), C.c_double(7.0), ptr(products), ptr(status))
    bytes_of = [torch.zeros(n * (width // 256) * 292, dtype=torch.uint8, device=gpu) for n in (rows, shared)]
    call("yvex_hip_q8k_quantize_swiglu", ptr(values), u64(rows), u64(width), ptr(bytes_of[0]), ptr(gate), ptr(up),
         u64(shared), C.c_double(7.0), ptr(bytes_of[1]), ptr(status))
    assert torch.equal(bytes_of[0], K.q8k_quantize(values, status))
    assert torch.equal(bytes_of[1], K.q8k_quantize(products, status)) and int(status.item()) == 0


@pytest.mark.parametrize("rows,width,gap", [(1, 256, 0), (3, 256, 1), (5, 768, 0), (7, 2304, 3), (9, 4096, 4)])
def test_four_blocks_a_wavefront_quantize_as_one_does(gpu, oracle, rows, width, gap):
    # blocks whose largest magnitude has both signs (the first decides), lies at an end, is zero, or so small that its inverse
    # is not finite (there only the kernel of one block a wavefront says what is right)
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"four.{rows}.{width}")
    x = np.asarray(g.normal(rows * width), dtype=np.float32).reshape(-1, 256)
    places = np.random.default_rng(rows).integers(0, 256, (x.shape[0], 2))
    for b in range(x.shape[0]):
        kind = b % 6
        if kind == 0:
            x[b] = -0.0 if b % 4 else 0.0
        elif kind in (1, 2):
            x[b, places[b, 0]], x[b, places[b, 1]] = 9.0, -9.0
        elif kind == 3:
            x[b] = np.where(np.arange(256) % 2 == b % 2, 1.0, -1.0)
        elif kind == 4:
            x[b, 255] = -11.0
    wide = torch.zeros((rows, width + gap), dtype=torch.float32, device=gpu)
    wide[:, :width] = dev(x.reshape(rows, width), gpu)
    status = K.new_status(gpu)
    got = torch.zeros(rows * (width // 256) * 292, dtype=torch.uint8, device=gpu)
    call("yvex_hip_q8k_quantize", ptr(wide), u64(rows), u64(width), u64(width + gap), ptr(got), ptr(status))
    assert np.array_equal(got.cpu().numpy(), oracle.q8k_quantize(x.reshape(rows, width))) and int(status.item()) == 0
    # tiny magnitudes and what is not finite, against the launch that takes a block a wavefront
    tiny = x.copy()
    tiny[::2] *= np.float32(1e-38)
    tiny = dev(tiny.reshape(rows, width), gpu)
    selected = torch.zeros((rows, 1), dtype=torch.int64, device=gpu)
    mine, encoded = K.Worklist(rows, 2, gpu), torch.empty_like(got)
    call("yvex_hip_moe_prepare_routed", ptr(selected), u64(rows), u64(2), u64(1), *K._wl_ptrs(mine), ptr(tiny), u64(width),
         u64(width), ptr(encoded), ptr(status))
    assert torch.equal(K.q8k_quantize(tiny, status), encoded) and int(status.item()) == 0
    for value in (float("inf"), float("nan")):
        broken, flag = tiny.clone(), K.new_status(gpu)
        broken[rows - 1, width - 1] = value
        K.q8k_quantize(broken, flag)
        assert int(flag.item()) == 1


@pytest.mark.parametrize("limit", [7.1, 40.1, 1.0e9])
def test_clamped_product_over_the_range_of_its_exponential(gpu, oracle, limit):
    # limits that binary32 does not hold, or arguments past 16, take the path in double; its exponential is within 0.6 units in
    # the last place of binary64, so that bfloat16 results are those of a correctly rounded one
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"swiglu.{limit}")
    gate = np.concatenate([np.asarray(g.normal(4096, spread), dtype=np.float32).reshape(-1) for spread in (1.0, 8.0, 40.0, 250.0)] +
                          [np.array([0.0, -0.0, 1e-30, -1e-30, -16.0, 16.0, -87.4, -708.5, -744.0, -746.0, -799.0, -801.0, -3e38, 3e38],
                                    dtype=np.float32)])
    up = np.asarray(g.normal(gate.size, 4.0), dtype=np.float32).reshape(-1)
    status = K.new_status(gpu)
    out = torch.empty(gate.size, dtype=torch.float32, device=gpu)
    held = dev(gate, gpu), dev(up, gpu)
    call("yvex_hip_moe_swiglu_rows", ptr(held[0]), ptr(held[1]), u64(gate.size), C.c_double(limit), ptr(out), ptr(status))
    gv = np.minimum(gate.astype(np.float64), limit)
    t = np.exp(-np.abs(gv))
    product = np.where(gv >= 0.0, gv / (1.0 + t), gv * t / (1.0 + t)) * np.clip(up.astype(np.float64), -limit, limit)
    with np.errstate(over="ignore"):
        want = torch.from_numpy(product.astype(np.float32)).to(torch.bfloat16).float()
    finite = torch.isfinite(want)
    assert same_bits(out.cpu()[finite], want[finite])
    assert int(status.item()) == (0 if bool(finite.all()) else 1)


# (the last: pair outputs that are loaded past the caches)
@pytest.mark.parametrize("rows,topk,width", [(1, 1, 4), (3, 6, 1028), (9, 8, 7168), (300, 8, 7172)])
def test_combine_goes_straight_into_the_egress(gpu, oracle, rows, topk, width):
    from yvex_amd import kernels as K
    streams = 4
    g = oracle.Generator(42, f"egress.{rows}.{width}")
    pairs = dev(g.normal(rows * topk * width).reshape(rows * topk, width), gpu)
    shared = dev(g.normal(rows * width).reshape(rows, width), gpu)
    x = dev(g.normal(rows * streams * width).reshape(rows, streams * width), gpu)
    post = dev(np.abs(g.normal(rows * streams)).reshape(rows, streams), gpu)
    mixing = dev(np.abs(g.normal(rows * 16)).reshape(rows, streams, streams), gpu)
    status = K.new_status(gpu)
    combined, routed = torch.empty_like(shared), torch.empty_like(shared)
    K.moe_reduce_combine(pairs, rows, topk, width, shared, routed, combined, status)
    want = K.mhc_egress(combined, x, post, mixing, streams=streams, width=width, status=status)
    got = torch.zeros_like(want)
    call("yvex_hip_moe_combine_egress", ptr(pairs), u64(rows), u64(topk), u64(streams), u64(width), ptr(shared), ptr(x),
         ptr(post), ptr(mixing), ptr(got), ptr(status))
    assert same_bits(got, want) and int(status.item()) == 0


@pytest.mark.parametrize("qtype,hidden,intermediate,experts,rows,topk", [
    ("IQ2_XXS", 2048, 2048, 3, 1, 3),          # a handful of iterations a workgroup, whole pieces of some empty
    ("IQ2_XXS", 7168, 2304, 9, 9, 5),          # one weight row an iteration, buckets of one to nine pairs
    ("Q4_K", 4096, 2048, 40, 16, 6)])
def test_sweeps_agree_with_the_matrix_core_kernels(gpu, oracle, qtype, hidden, intermediate, experts, rows, topk):
    """Wherever a workgroup's piece of the launch begins and ends, the sweeps publish what the matrix-core
    kernels publish for the same worklist (both are the CPU path's bits)."""
    from yvex_amd import kernels as K
    qt = getattr(oracle, qtype)
    g = oracle.Generator(42, f"pieces.{qtype}.{hidden}.{experts}")
    tensors = [dev(g.weights(qt, experts * r, w), gpu) for r, w in
               ((intermediate, hidden), (intermediate, hidden), (hidden, intermediate))]
    weights = K.expert_weights(*tensors, (qt, qt, qt), hidden, intermediate)
    status = K.new_status(gpu)
    logits = dev(g.normal(rows * experts).reshape(rows, experts) - 0.35 * np.arange(experts), gpu)
    selected, route = K.moe_route_rows(logits.float(), None, topk, K.SIGMOID, True, 1.0, status)
    wl, pairs = K.worklist_build(selected, experts, status), rows * topk
    act = K.q8k_quantize(dev(g.normal(rows * hidden).reshape(rows, hidden), gpu), status)
    mid = [torch.zeros((pairs, intermediate), device=gpu) for _ in range(2)]
    K.moe_up(weights, act, True, route, wl, pairs, topk, experts, 10.0, mid[0], status)
    K.moe_up_rows(weights, act, route, wl, pairs, topk, experts, 10.0, mid[1], status)
    assert same_bits(mid[0], mid[1])
    mid_q8 = K.q8k_quantize(mid[0], status)
    out = [torch.zeros((pairs, hidden), device=gpu) for _ in range(2)]
    K.moe_down(weights, mid_q8, True, wl, pairs, experts, out[0], status)
    K.moe_down_rows(weights, mid_q8, wl, pairs, experts, out[1], status)
    assert same_bits(out[0], out[1]) and int(status.item()) == 0


# selections that a thread keeps and that it reads again, the order put together in LDS and stored word by word, with and
# without the table of counts below a word; one row, one expert, a selection that repeats or is no expert
@pytest.mark.parametrize("rows,experts,topk,fault", [
    (1, 1, 1, None), (513, 256, 8, None), (2048, 256, 8, None), (2047, 256, 9, None), (3001, 250, 6, None), (4096, 256, 8, None),
    (4096, 7, 7, None), (1111, 33, 3, "twice"), (1111, 33, 3, "none")])
def test_worklist_and_quantization_in_one_launch(gpu, oracle, rows, experts, topk, fault):
    from yvex_amd import kernels as K
    width, g = 512, oracle.Generator(42, f"large.worklist.{rows}.{experts}.{topk}")
    keys = g.normal(rows * experts).reshape(rows, experts) - 0.05 * np.arange(experts)
    chosen = np.argsort(-keys, axis=1)[:, :topk].astype(np.int64)
    if fault:
        chosen[700, 2] = chosen[700, 0] if fault == "twice" else experts
    selected, x = dev(chosen, gpu), dev(g.normal(rows * width).reshape(rows, width), gpu)
    status = [K.new_status(gpu) for _ in range(2)]
    wl, q8 = [K.Worklist(rows * topk, experts, gpu) for _ in range(2)], [torch.zeros(rows * 2 * 292, dtype=torch.uint8, device=gpu)] * 2
    K.worklist_build(selected, experts, status[0], wl[0])
    q8[0] = K.q8k_quantize(x, status[0]).view(torch.uint8).reshape(-1)
    call("yvex_hip_worklist_quantize", ptr(selected), u64(rows * topk), u64(topk), u64(experts), ptr(wl[1].order),
         ptr(wl[1].expert_ids), ptr(wl[1].bucket_offsets), ptr(wl[1].bucket_populations), ptr(wl[1].sweep_offsets),
         ptr(wl[1].counts), ptr(x), u64(width), ptr(q8[1]), ptr(status[1]))
    assert torch.equal(q8[0], q8[1]) and [int(s.item()) for s in status] == [2 if fault else 0] * 2
    if fault:
        return
    for name in ("order", "expert_ids", "bucket_populations", "counts"):
        assert torch.equal(getattr(wl[0], name), getattr(wl[1], name)), name
    buckets = int(wl[0].counts[0].item())
    assert torch.equal(wl[0].order, torch.sort(selected.reshape(-1), stable=True)[1])
    for name in ("bucket_offsets", "sweep_offsets"):
        assert torch.equal(getattr(wl[0], name)[:buckets + 1], getattr(wl[1], name)[:buckets + 1]), name


# so many choices a row that a row number by multiplication comes out one too high for the last pair: of 32 (96) rows that is the
# first bit of another expert's words
@pytest.mark.parametrize("rows,topk", [(32, 11627), (96, 6733)])
def test_more_choices_a_row_than_experts_reach_no_other_experts_words(gpu, rows, topk):
    """Such a batch repeats experts and is refused; its lists hold the rows that chose an expert and nothing else."""
    from yvex_amd import kernels as K
    experts, width, pairs = 9, 256, rows * topk
    inverse = 0xffffffff // topk + 1
    assert ((pairs - 1) * inverse >> 32) == rows and (rows // 32) % 2 == 1
    selected, x = torch.full((rows, topk), 5, dtype=torch.int64, device=gpu), torch.ones((rows, width), device=gpu)
    q8 = torch.zeros(rows * 292, dtype=torch.uint8, device=gpu)
    for quantizing in (False, True):
        wl, status = K.Worklist(pairs, experts, gpu), K.new_status(gpu)
        wl.order.zero_()
        if quantizing:
            call("yvex_hip_worklist_quantize", ptr(selected), u64(pairs), u64(topk), u64(experts), *K._wl_ptrs(wl), ptr(x),
                 u64(width), ptr(q8), ptr(status))
        else:
            K.worklist_build(selected, experts, status, wl)
        assert int(status.item()) == 2
        assert wl.counts.tolist()[:3] == [1, rows, rows] and wl.expert_ids[0].item() == 5
        assert wl.bucket_populations.tolist() == [rows] + [0] * (experts - 1)
        assert bool(((wl.order >= 0) & (wl.order < pairs)).all())


# ranks in one batch of loads and in several, columns in fours and one by one, edges of a workgroup's columns, more rows
# than a grid has in its second direction, outputs that are loaded past the caches
@pytest.mark.parametrize("rows,topk,hidden", [(1, 1, 4), (3, 8, 1024), (2, 9, 1028), (5, 17, 258), (1, 6, 2050), (65537, 2, 4), (2100, 8, 1028)])
def test_reduce_adds_ranks_in_order(gpu, oracle, rows, topk, hidden):
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"reduce.{rows}.{topk}.{hidden}")
    pairs = dev(g.normal(rows * topk * hidden).reshape(rows, topk, hidden).astype(np.float32), gpu)
    shared = dev(g.normal(rows * hidden).reshape(rows, hidden).astype(np.float32), gpu)
    routed, combined, status = torch.zeros_like(shared), torch.zeros_like(shared), K.new_status(gpu)
    K.moe_reduce_combine(pairs, rows, topk, hidden, shared, routed, combined, status)
    want = torch.zeros_like(shared)
    for rank in range(topk):
        want += pairs[:, rank]
    assert same_bits(routed, want) and same_bits(combined, (want + shared).to(torch.bfloat16).float()) and int(status.item()) == 0
    pairs[rows - 1, topk - 1, hidden - 1] = float("nan")
    K.moe_reduce_combine(pairs, rows, topk, hidden, shared, routed, combined, status)
    assert int(status.item()) == 1


# a shared tile of one row, a whole one, one and a row; few routed pairs and several tiles a bucket; with the few-pair
# kernels beside (1100 rows of two superblocks, which a matrix alone has too many of for them)
@pytest.mark.parametrize("down,hidden,intermediate,rows,topk", [
    ("Q4_K", 256, 256, 1, 2), ("Q4_K", 256, 256, 64, 1), ("Q2_K", 256, 256, 65, 3), ("Q2_K", 256, 256, 200, 3),
    ("Q4_K", 1024, 512, 1100, 2)])
def test_shared_rows_join_the_routed_launch(gpu, oracle, down, hidden, intermediate, rows, topk):
    """One launch writes what the two it replaces write, bit for bit; an unsuitable pair is refused."""
    from yvex_amd import kernels as K
    experts, g = 7, oracle.Generator(42, f"join.{down}.{hidden}.{intermediate}.{rows}")
    kinds = (oracle.Q4_K, oracle.Q4_K, getattr(oracle, down))
    shapes = ((intermediate, hidden), (intermediate, hidden), (hidden, intermediate))
    routed, shared = (K.expert_weights(*(dev(g.weights(qt, n * r, w), gpu) for qt, (r, w) in zip(kinds, shapes)), kinds, hidden,
                                       intermediate) for n in (experts, 1))
    status = K.new_status(gpu)
    logits = dev(g.normal(rows * experts).reshape(rows, experts) - 0.5 * np.arange(experts), gpu)
    selected, route = K.moe_route_rows(logits.float(), None, topk, K.SIGMOID, True, 1.0, status)
    wl, pairs = K.worklist_build(selected, experts, status), rows * topk
    act = K.q8k_quantize(dev(g.normal(rows * hidden).reshape(rows, hidden), gpu), status)
    assert all(K.moe_rows_join(routed, wl, pairs, topk, experts, shared, rows, way) for way in (0, 1))
    mid, mid_shared = ([torch.zeros((n, intermediate), device=gpu) for _ in range(2)] for n in (pairs, rows))
    K.moe_up_rows(routed, act, route, wl, pairs, topk, experts, 10.0, mid[0], status)
    K.moe_up_rows(shared, act, None, None, rows, 1, 1, 10.0, mid_shared[0], status)
    K.moe_up_rows_joined(routed, act, route, wl, pairs, topk, experts, 10.0, mid[1], shared, rows, mid_shared[1], status)
    assert same_bits(mid[0], mid[1]) and same_bits(mid_shared[0], mid_shared[1]) and bool(mid_shared[0].any())
    mid_q8, shared_q8 = K.q8k_quantize(mid[0], status), K.q8k_quantize(mid_shared[0], status)
    out, out_shared = ([torch.zeros((n, hidden), device=gpu) for _ in range(2)] for n in (pairs, rows))
    K.moe_down_rows(routed, mid_q8, wl, pairs, experts, out[0], status)
    K.moe_down_rows(shared, shared_q8, None, rows, 1, out_shared[0], status)
    K.moe_down_rows_joined(routed, mid_q8, wl, pairs, experts, out[1], shared, shared_q8, rows, out_shared[1], status)
    assert same_bits(out[0], out[1]) and same_bits(out_shared[0], out_shared[1]) and bool(out_shared[0].any())
    assert int(status.item()) == 0
    other = K.expert_weights(*shared._keep, (oracle.Q4_K, oracle.Q4_K, oracle.IQ2_XXS), hidden, intermediate)
    assert not K.moe_rows_join(routed, wl, pairs, topk, experts, other, rows, 1)
    with pytest.raises(Exception):
        K.moe_down_rows_joined(routed, mid_q8, wl, pairs, experts, out[1], other, shared_q8, rows, out_shared[1], status)


# a pair, a remainder of the largest size the few-pair kernels take at the width and one more, 64-pair
# tiles with and without such remainders; two, three and 32 superblocks a row, ragged row units
@pytest.mark.parametrize("up,down,hidden,intermediate,tokens,image", [
    ("IQ2_XXS", "Q2_K", 1024, 768, 16, True), ("IQ2_XXS", "IQ2_XXS", 7168, 512, 12, True),
    ("IQ2_XXS", "IQ2_XXS", 7168, 512, 12, False), ("IQ2_XXS", "IQ2_XXS", 512, 1024, 16, False),
    ("Q4_K", "Q4_K", 768, 1024, 16, False), ("Q4_K", "Q2_K", 7168, 512, 16, False),
    ("IQ2_XXS", "Q4_K", 8192, 256, 8, True), ("IQ2_XXS", "Q2_K", 512, 2304, 16, True)])
def test_few_pair_kernels_agree_with_the_generic_kernel(gpu, oracle, up, down, hidden, intermediate, tokens, image):
    """Buckets split between the two row-batch kernels by their remainders, and a matrix alone, hold
    what the generic grouped kernel (the CPU path's bits) publishes for the same pairs."""
    from yvex_amd import kernels as K
    uq, dq = getattr(oracle, up), getattr(oracle, down)
    populations = [1, tokens, tokens + 1, 64 + tokens, 64, 0, 64 + tokens + 1, 5]
    experts, pairs = len(populations), sum(populations)
    g = oracle.Generator(43, f"few.{up}.{down}.{hidden}")
    tensors = [dev(g.weights(q, experts * r, w), gpu) for q, r, w in
               ((uq, intermediate, hidden), (uq, intermediate, hidden), (dq, hidden, intermediate))]
    weights = K.expert_weights(*tensors, (uq, uq, dq), hidden, intermediate)
    rows_form = K.expert_weights(*tensors, (uq, uq, dq), hidden, intermediate)
    images = [K.iq2_sweep_image(t) if image and q == oracle.IQ2_XXS else None for t, q in zip(tensors, (uq, uq, dq))]
    if images[0] is not None:
        rows_form.gate, rows_form.up, rows_form.gate_up_image = images[0].data_ptr(), images[1].data_ptr(), 1
        rows_form.gate_row_bytes = rows_form.up_row_bytes = hidden // 256 * 72
        rows_form.gate_expert_bytes = rows_form.up_expert_bytes = hidden // 256 * 72 * intermediate
    if images[2] is not None:
        rows_form.down, rows_form.down_image = images[2].data_ptr(), 1
        rows_form.down_row_bytes, rows_form.down_expert_bytes = intermediate // 256 * 72, intermediate // 256 * 72 * hidden
    status = K.new_status(gpu)
    selected = torch.repeat_interleave(torch.arange(experts), torch.tensor(populations))
    selected = selected[torch.randperm(pairs, generator=torch.Generator().manual_seed(3))].reshape(pairs, 1).to(gpu)
    wl = K.worklist_build(selected, experts, status)
    route = dev((0.5 + np.abs(g.normal(pairs))).astype(np.float32), gpu)
    act = K.q8k_quantize(dev(g.normal(pairs * hidden).reshape(pairs, hidden), gpu), status)
    mid = [torch.zeros((pairs, intermediate), device=gpu) for _ in range(2)]
    K.moe_up(weights, act, True, route, wl, pairs, 1, experts, 10.0, mid[0], status)
    K.moe_up_rows(rows_form, act, route, wl, pairs, 1, experts, 10.0, mid[1], status)
    assert same_bits(mid[0], mid[1])
    mid_q8 = K.q8k_quantize(mid[0], status)
    out = [torch.zeros((pairs, hidden), device=gpu) for _ in range(2)]
    K.moe_down(weights, mid_q8, True, wl, pairs, experts, out[0], status)
    K.moe_down_rows(rows_form, mid_q8, wl, pairs, experts, out[1], status)
    assert same_bits(out[0], out[1])
    for alone in (tokens + 3, 257):                     # one matrix for all rows
        some = K.q8k_quantize(dev(g.normal(alone * hidden).reshape(alone, hidden), gpu), status)
        mid = [torch.zeros((alone, intermediate), device=gpu) for _ in range(2)]
        K.moe_up(weights, some, True, None, None, alone, 1, 1, 10.0, mid[0], status)
        K.moe_up_rows(rows_form, some, None, None, alone, 1, 1, 10.0, mid[1], status)
        assert same_bits(mid[0], mid[1])
    assert int(status.item()) == 0


# one more pair than a tile of the few-pair kernels, two tiles' pairs, one more; as many such buckets as their second tiles
# are for and one more; rows of four, five and 28 superblocks (two at a time, one, one and twelve pairs a tile)
@pytest.mark.parametrize("hidden,intermediate,tokens", [(1024, 1024, 16), (1280, 512, 16), (7168, 256, 12)])
@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("tail", ["within", "beyond"])
def test_few_pair_kernels_take_second_tiles(gpu, oracle, hidden, intermediate, tokens, extra, tail):
    """What the 64-pair kernels leave and the few-pair kernels take is each pair once, whichever side of
    the rule for second tiles a batch is on."""
    from yvex_amd import kernels as K
    uq, dq = oracle.IQ2_XXS, oracle.Q2_K
    populations = [tokens + 1 + (i * 3) % tokens for i in range(16 + extra)] + [2 * tokens + (tail == "beyond"), 1, tokens]
    populations = populations[1:]                       # sixteen buckets past a tile, or seventeen
    experts, pairs = len(populations), sum(populations)
    g = oracle.Generator(44, f"second.{hidden}")
    tensors = [dev(g.weights(q, experts * r, w), gpu) for q, r, w in
               ((uq, intermediate, hidden), (uq, intermediate, hidden), (dq, hidden, intermediate))]
    weights = K.expert_weights(*tensors, (uq, uq, dq), hidden, intermediate)
    rows_form = K.expert_weights(*tensors, (uq, uq, dq), hidden, intermediate)
    images = [K.iq2_sweep_image(t) for t in tensors[:2]]
    rows_form.gate, rows_form.up, rows_form.gate_up_image = images[0].data_ptr(), images[1].data_ptr(), 1
    rows_form.gate_row_bytes = rows_form.up_row_bytes = hidden // 256 * 72
    rows_form.gate_expert_bytes = rows_form.up_expert_bytes = hidden // 256 * 72 * intermediate
    status = K.new_status(gpu)
    selected = torch.repeat_interleave(torch.arange(experts), torch.tensor(populations)).reshape(pairs, 1).to(gpu)
    wl = K.worklist_build(selected, experts, status)
    route = dev((0.5 + np.abs(g.normal(pairs))).astype(np.float32), gpu)
    act = K.q8k_quantize(dev(g.normal(pairs * hidden).reshape(pairs, hidden), gpu), status)
    mid = [torch.full((pairs, intermediate), float("nan"), device=gpu) for _ in range(2)]
    K.moe_up(weights, act, True, route, wl, pairs, 1, experts, 10.0, mid[0], status)
    K.moe_up_rows(rows_form, act, route, wl, pairs, 1, experts, 10.0, mid[1], status)
    assert same_bits(mid[0], mid[1])
    mid_q8 = K.q8k_quantize(mid[0], status)
    out = [torch.full((pairs, hidden), float("nan"), device=gpu) for _ in range(2)]
    K.moe_down(weights, mid_q8, True, wl, pairs, experts, out[0], status)
    K.moe_down_rows(rows_form, mid_q8, wl, pairs, experts, out[1], status)
    assert same_bits(out[0], out[1]) and int(status.item()) == 0


# more row tiles than workgroups, so that pieces begin and end inside token tiles and pass from tiles of 64 pairs to ones of 33 to
# 63 and of fewer than 33; rows of an odd number of superblocks, of two and of many
@pytest.mark.parametrize("hidden,intermediate", [(8192, 512), (1280, 4096)])
@pytest.mark.parametrize("image", [True, False])
def test_runs_of_row_tiles_agree_with_the_sweeps(gpu, oracle, hidden, intermediate, image):
    """A workgroup of the 64-pair kernel goes from row tile to row tile and from token tile to token tile: each pair's rows
    come out once, the sweeps' bits."""
    from yvex_amd import kernels as K
    qt, populations = oracle.IQ2_XXS, [420, 33, 260, 130, 20, 100, 64, 29]
    experts, pairs = len(populations), sum(populations)
    g = oracle.Generator(45, f"runs.{hidden}")
    tensors = [dev(g.weights(qt, experts * r, w), gpu) for r, w in
               ((intermediate, hidden), (intermediate, hidden), (hidden, intermediate))]
    weights = K.expert_weights(*tensors, (qt, qt, qt), hidden, intermediate)
    rows_form = K.expert_weights_image(weights, hidden, intermediate) if image else weights
    status = K.new_status(gpu)
    selected = torch.repeat_interleave(torch.arange(experts), torch.tensor(populations))
    selected = selected[torch.randperm(pairs, generator=torch.Generator().manual_seed(5))].reshape(pairs, 1).to(gpu)
    wl = K.worklist_build(selected, experts, status)
    route = dev((0.5 + np.abs(g.normal(pairs))).astype(np.float32), gpu)
    act = K.q8k_quantize(dev(g.normal(pairs * hidden).reshape(pairs, hidden), gpu), status)
    mid = [torch.full((pairs, intermediate), float("nan"), device=gpu) for _ in range(2)]
    K.moe_up(weights, act, True, route, wl, pairs, 1, experts, 10.0, mid[0], status)
    K.moe_up_rows(rows_form, act, route, wl, pairs, 1, experts, 10.0, mid[1], status)
    assert same_bits(mid[0], mid[1])
    mid_q8 = K.q8k_quantize(mid[0], status)
    out = [torch.full((pairs, hidden), float("nan"), device=gpu) for _ in range(2)]
    K.moe_down(weights, mid_q8, True, wl, pairs, experts, out[0], status)
    K.moe_down_rows(rows_form, mid_q8, wl, pairs, experts, out[1], status)
    assert same_bits(out[0], out[1]) and int(status.item()) == 0


def packed_iq2(rows, width, seed, device):
    """Random IQ2_XXS rows: any codes, small positive scales."""
    gen = torch.Generator(device=device).manual_seed(seed)
    raw = torch.empty((rows * width // 256, 66), dtype=torch.uint8, device=device).random_(generator=gen)
    scale = torch.rand((raw.shape[0], 1), generator=gen, device=device).mul_(2.5e-4).add_(1e-4).to(torch.float16)
    raw[:, :2] = scale.view(torch.uint8)
    return raw.reshape(-1)


# long tiles enough for some workgroups only, and for every one; the short ones (17 to 32 pairs, which the few-pair kernels
# leave to this one) make up the difference; odd numbers of superblocks and row tiles
@pytest.mark.parametrize("long_ones", [[64, 40, 128, 63, 200], [64, 33] * 12 + [128, 50] * 6], ids=["few", "many"])
@pytest.mark.parametrize("image", [True, False], ids=["image", "canonical"])
def test_short_tiles_fill_up_the_shares_of_long_ones(gpu, oracle, long_ones, image):
    """The 64-pair IQ2_XXS kernel deals long and short tiles out separately where there are short ones enough: every pair's rows
    come out once, the sweeps' bits."""
    from yvex_amd import kernels as K
    hidden, intermediate, qt = 2304, 1280, oracle.IQ2_XXS
    populations = [n for pair in zip(long_ones + [0] * 48, [17 + k % 16 for k in range(48)]) for n in pair if n]
    experts, pairs = len(populations), sum(populations)
    grid = torch.cuda.get_device_properties(gpu).multi_processor_count
    for out_rows, tile in ((intermediate, 128), (hidden, 256)):
        tiles = out_rows // tile
        wide = tiles * sum(n // 64 + (n % 64 > 32) for n in populations)
        narrow = tiles * sum(17 <= n % 64 <= 32 for n in populations)
        assert (4 * wide + 3 * narrow) // grid >= 4 * (wide // grid + 1), "long and short tiles are not dealt out separately here"
    tensors = [packed_iq2(experts * r, w, 7 + k, gpu) for k, (r, w) in
               enumerate(((intermediate, hidden), (intermediate, hidden), (hidden, intermediate)))]
    weights = K.expert_weights(*tensors, (qt, qt, qt), hidden, intermediate)
    rows_form = K.expert_weights_image(weights, hidden, intermediate) if image else weights
    status, g = K.new_status(gpu), oracle.Generator(47, f"shares.{experts}")
    selected = torch.repeat_interleave(torch.arange(experts), torch.tensor(populations))
    selected = selected[torch.randperm(pairs, generator=torch.Generator().manual_seed(6))].reshape(pairs, 1).to(gpu)
    wl = K.worklist_build(selected, experts, status)
    route = dev((0.5 + np.abs(g.normal(pairs))).astype(np.float32), gpu)
    act = K.q8k_quantize(dev(g.normal(pairs * hidden).reshape(pairs, hidden), gpu), status)
    mid = [torch.full((pairs, intermediate), float("nan"), device=gpu) for _ in range(2)]
    K.moe_up(weights, act, True, route, wl, pairs, 1, experts, 10.0, mid[0], status)
    K.moe_up_rows(rows_form, act, route, wl, pairs, 1, experts, 10.0, mid[1], status)
    assert bool(torch.isfinite(mid[0]).all()) and same_bits(mid[0], mid[1])
    mid_q8 = K.q8k_quantize(mid[0], status)
    out = [torch.full((pairs, hidden), float("nan"), device=gpu) for _ in range(2)]
    K.moe_down(weights, mid_q8, True, wl, pairs, experts, out[0], status)
    K.moe_down_rows(rows_form, mid_q8, wl, pairs, experts, out[1], status)
    assert bool(torch.isfinite(out[0]).all()) and same_bits(out[0], out[1]) and int(status.item()) == 0


# a last row tile of four rows and of 252, one superblock and an odd number of them
@pytest.mark.parametrize("rows,width,inputs", [(4100, 1280, 2048), (7164, 256, 1025)])
def test_ragged_row_tiles_run_alone(gpu, oracle, rows, width, inputs):
    """A projection whose last row tile is not whole holds what the kernels of a few input rows publish."""
    from yvex_amd import kernels as K
    qt = oracle.IQ2_XXS
    g = oracle.Generator(46, f"ragged.{rows}")
    weights, status = dev(g.weights(qt, rows, width), gpu), K.new_status(gpu)
    act = K.q8k_quantize(dev(g.normal(inputs * width).reshape(inputs, width), gpu), status)
    got = K.matvec(weights, qt, rows, width, act, input_q8=True, input_rows=inputs, status=status)
    stride = width // 256 * 292
    for at in (0, 61, inputs - 5):
        few = K.matvec(weights, qt, rows, width, act[at * stride:(at + 5) * stride].contiguous(), input_q8=True, input_rows=5,
                       status=status)
        assert same_bits(got[at:at + 5], few)
    assert int(status.item()) == 0


# 16, 32 and 64 input rows a workgroup of the staged kernel (on 256 compute units), ragged on both sides,
# one chunk and several
@pytest.mark.parametrize("rows,width,inputs", [(250, 384, 345), (256, 128, 850), (249, 256, 2045)])
def test_router_blocks_of_every_size_are_sums_in_double(gpu, rows, width, inputs):
    from yvex_amd import kernels as K
    gen = torch.Generator().manual_seed(rows)
    w, x = torch.randn((rows, width), generator=gen), torch.randn((inputs, width), generator=gen)
    status = K.new_status(gpu)
    got = K.matvec(w.to(gpu).view(torch.uint8), 0, rows, width, x.to(gpu), status=status).cpu()
    want = (x.double() @ w.double().t()).float()
    # sums in double in another order differ by under 1e-13 of the terms: the float is the same or, next
    # to a rounding boundary, its neighbour
    assert torch.all((got - want).abs() <= want.abs() * 2.0 ** -23 + 1e-12) and int(status.item()) == 0


# a row below and at the line between the sweeps and the tiles: the constant part and the cap of each rule
@pytest.mark.parametrize("qtype,shared,hidden,experts,at", [
    ("IQ2_XXS", True, 512, 8, 62), ("IQ2_XXS", True, 512, 4, 36), ("IQ2_XXS", True, 5632, 8, 53), ("IQ2_XXS", "Q8_0", 512, 16, 41),
    ("IQ2_XXS", False, 512, 8, 24), ("Q4_K", True, 512, 24, 45), ("Q4_K", True, 512, 4, 8), ("Q4_K", False, 512, 8, 11)])
def test_row_batches_either_side_of_the_matrix_core_line(gpu, oracle, qtype, shared, hidden, experts, at):
    from backend_helpers import Backend
    from test_gpu_backend import MoeCase, same_as_cpu
    for rows in (at - 1, at):
        b = Backend()
        try:
            case = MoeCase(b, oracle, qtype=qtype, hidden=hidden, experts=experts, topk=2, rows=rows, shared=bool(shared),
                           shared_qtype=shared if isinstance(shared, str) else None)
            b.workspace(case.workspace_bytes)
            assert case.execute() == 0, case.err.message
            assert (case.result.tensor_core_launches > 0) == (rows == at)
            want = case.oracle_layer(act_q8=True)
            assert np.array_equal(case.sel.reshape(rows, 2), want["selected"])
            same_as_cpu(case.combined, want["combined"])
        finally:
            assert b.close() == 0


# the layer as a decoder runs it, deferred and without host copies, whose combine goes straight into the egress; the
# caller alternates with batches that ask for host copies, each kind eager, captured and replayed; the last is the widest row
# of a layer, by as many rows as the ingress needs to join its projection
@pytest.mark.parametrize("down,shared,rows,width", [(None, None, 1, 512), ("Q2_K", "Q8_0", 5, 512), ("Q2_K", "Q8_0", 75, 512),
                                                    (None, None, 8, 8192)])
def test_deferred_layers_with_streams_are_the_oracles(gpu, oracle, down, shared, rows, width):
    from backend_helpers import Backend
    from test_gpu_backend import MoeCase, same_as_cpu
    from yvex_amd import abi
    b = Backend()
    try:
        case = MoeCase(b, oracle, hidden=width, intermediate=512, rows=rows, streams=4, down_qtype=down, shared_qtype=shared)
        b.workspace(case.workspace_bytes)
        want, host, done = case.oracle_layer(act_q8=True), case.out, abi.RowBatchResult()
        empty, zeros = abi.RowBatchOutput(), np.zeros_like(case.x)
        completion = abi.DeviceCompletion(1, None)
        for sight in range(3):
            for kind in ("host copies", "deferred", "no copies"):
                assert b.lib.yvex_rocm_backend_tensor_write(b.handle, case.rows_out, zeros.ctypes.data, zeros.nbytes,
                                                            C.byref(case.err)) == 0
                case.combined.fill(0.0)
                case.out = host if kind == "host copies" else empty
                case.job.device_completion = C.pointer(completion) if kind == "deferred" else None
                assert case.execute() == 0, case.err.message
                if kind == "deferred":
                    assert case.ops.complete_rows(b.handle, 0, C.byref(done), C.byref(case.err)) == 0, case.err.message
                # (deferred or not, batches without host copies are one topology)
                assert case.result.graph_replays == (sight == 2 or (sight == 1 and kind != "host copies"))
                if kind == "host copies":
                    assert np.max(np.abs(case.post - want["post"])) <= 1e-6
                    assert np.max(np.abs(case.comb - want["combination"])) <= 1e-6
                    same_as_cpu(case.combined, want["combined"])
                    # the egress of the CPU's combined rows with the device's own gates is exact
                    rc, egress = oracle.mhc_post(want["combined"], case.x, case.post, case.comb, streams=4, width=width)
                    assert rc == 0
                else:
                    assert not case.combined.any()
                got = b.read_f32(case.rows_out, case.x.size).reshape(case.x.shape)
                assert np.array_equal(got.view(np.uint32), egress.view(np.uint32)), kind
    finally:
        assert b.close() == 0


# matrices past 32 768 rows against few input rows: one round of the 16-token tiles, and more than one
@pytest.mark.parametrize("rows,inputs", [(32772, 8), (50004, 17), (99332, 9)])
def test_iq2_rows_of_tall_matrices_are_the_sweeps_bits(gpu, oracle, rows, inputs):
    from yvex_amd import kernels as K
    width = 512
    g = oracle.Generator(44, f"tall.{rows}")
    w = dev(g.weights(oracle.IQ2_XXS, rows, width), gpu)
    x = dev(g.normal(inputs * width).reshape(inputs, width), gpu)
    status = K.new_status(gpu)
    got = K.matvec(w, oracle.IQ2_XXS, rows, width, K.q8k_quantize(x, status), input_q8=True, input_rows=inputs, status=status)
    for at in range(0, inputs, 7):                     # (fewer than eight input rows: the sweep)
        some = x[at:at + 7].contiguous()
        want = K.matvec(w, oracle.IQ2_XXS, rows, width, K.q8k_quantize(some, status), input_q8=True,
                        input_rows=some.shape[0], status=status)
        assert same_bits(got[at:at + 7], want)
    assert int(status.item()) == 0


# the 32-row tiles of the F32 projection: ragged on both sides, fewer columns than waves, one launch and split, 16 and 32
# input rows a tile; formats other than F32 (one launch); below eight input rows, sixteen waves a weight row
@pytest.mark.parametrize("qtype,rows,width,inputs", [
    ("F32", 1, 128, 257), ("F32", 250, 1024, 1570), ("F32", 33, 16512, 17), ("F32", 65, 2176, 301), ("F32", 255, 4096, 97),
    ("F32", 200, 6148, 5), ("F32", 129, 6400, 6), ("F32", 250, 7168, 7), ("F32", 24, 16388, 7), ("F32", 3, 33000, 2),
    ("F16", 31, 64, 256), ("BF16", 33, 320, 511), ("Q8_0", 97, 448, 289)])
def test_f32_tiles_of_32_weight_rows_match_float64(gpu, oracle, qtype, rows, width, inputs):
    """Sums of exact products in double, rounded once: half a unit in the last place and the double
    sums' own error, which a sum of `width` terms bounds by width 2^-52 of the terms' magnitudes."""
    from yvex_amd import kernels as K
    qt = getattr(oracle, qtype)
    g = oracle.Generator(42, f"tile32.{qtype}.{rows}.{width}.{inputs}")
    x = g.normal(inputs * width).reshape(inputs, width)
    if qtype in ("F16", "BF16"):
        half = torch.from_numpy(g.normal(rows * width)).to(torch.float16 if qtype == "F16" else torch.bfloat16)
        w = half.view(torch.uint8).numpy()
    else:
        w = g.weights(qt, rows, width)
    values = oracle.decode_rows(qt, w, width).reshape(rows, width).astype(np.float64)
    status = K.new_status(gpu)
    want = x.astype(np.float64) @ values.T
    slack = np.abs(want) * 2.0 ** -24 + width * 2.0 ** -52 * (np.abs(x.astype(np.float64)) @ np.abs(values).T)
    one = K.matvec(dev(w, gpu), qt, rows, width, dev(x, gpu), status=status).cpu().numpy()
    assert np.all(np.abs(one - want) <= slack)
    if qtype == "F32":
        split = K.matvec_f32_rows(dev(w.view(np.float32).reshape(rows, width), gpu), dev(x, gpu), status).cpu().numpy()
        assert np.all(np.abs(split - want) <= slack)
    assert int(status.item()) == 0


# one input tile's workgroups test the weights for all: one input tile and several, of both sizes
@pytest.mark.parametrize("inputs", [8, 40, 1500])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_a_weight_that_is_no_number_is_reported_once_for_all_input_rows(gpu, inputs, value):
    from yvex_amd import kernels as K
    weights, x = torch.ones((70, 1024), device=gpu), torch.ones((inputs, 1024), device=gpu)
    for row, column in ((0, 0), (37, 1023), (69, 500)):
        held, status = weights.clone(), K.new_status(gpu)
        assert bool((K.matvec_f32_rows(held, x, status) == 1024.0).all()) and int(status.item()) == 0
        held[row, column] = value
        K.matvec_f32_rows(held, x, status)
        assert int(status.item()) == 1


# the shared expert's Q8_0 products beside preparation and quantization: the separate launches' bits, at one and two rows,
# fewer weight rows than a workgroup has waves, rows between dword boundaries, several rows a wave
@pytest.mark.parametrize("rows,hidden,middle,experts,topk,offset", [(1, 256, 256, 4, 2, 0), (2, 2048, 768, 16, 4, 2),
                                                                    (1, 7168, 2048, 256, 8, 0), (2, 4352, 5120, 33, 3, 2)])
def test_shared_products_ride_along(gpu, oracle, rows, hidden, middle, experts, topk, offset):
    from yvex_amd import kernels as K
    g = oracle.Generator(42, f"ride.{rows}.{hidden}.{middle}")
    lib, Q = K.load_library(), oracle.Q8_0

    def matrix(n, width):
        held = torch.zeros(n * width // 32 * 34 + offset, dtype=torch.uint8, device=gpu)
        held[offset:] = dev(g.weights(Q, n, width), gpu)
        return held[offset:]
    gate, up, down = matrix(middle, hidden), matrix(middle, hidden), matrix(hidden, middle)
    x = dev(g.normal(rows * hidden).reshape(rows, hidden), gpu)
    logits = dev(g.normal(rows * experts).reshape(rows, experts), gpu)
    routed = dev(g.normal(rows * topk * middle).reshape(rows * topk, middle), gpu)
    status = K.new_status(gpu)
    wl = K.Worklist(rows * topk, experts, gpu)
    q8 = torch.zeros(rows * (hidden // 256) * 292, dtype=torch.uint8, device=gpu)
    sel, weights = K.moe_prepare(logits, None, topk, K.SIGMOID, True, 1.5, status, wl, x, q8)
    want = [K.matvec(w, Q, middle, hidden, q8, input_q8=True, input_rows=rows, status=status) for w in (gate, up)]
    mid = [torch.zeros(n * (middle // 256) * 292, dtype=torch.uint8, device=gpu) for n in (rows * topk, rows)]
    limit = 3.0
    call("yvex_hip_q8k_quantize_swiglu", ptr(routed), u64(rows * topk), u64(middle), ptr(mid[0]), ptr(want[0]), ptr(want[1]),
         u64(rows), C.c_double(limit), ptr(mid[1]), ptr(status))
    want_down = K.matvec(down, Q, hidden, middle, mid[1], input_q8=True, input_rows=rows, output_bf16=True, status=status)

    class Pair(C.Structure):
        _fields_ = [("first", C.c_void_p), ("second", C.c_void_p), ("row_count", C.c_uint64), ("row_bytes", C.c_uint64),
                    ("out_first", C.c_void_p), ("out_second", C.c_void_p)]
    got = [torch.full((rows, middle), 7.0, device=gpu) for _ in range(2)]
    pair = Pair(gate.data_ptr(), up.data_ptr(), middle, hidden // 32 * 34, got[0].data_ptr(), got[1].data_ptr())
    assert lib.yvex_hip_moe_prepare_projecting_supported(C.byref(pair), u64(rows), u64(hidden))
    wl2, q82 = K.Worklist(rows * topk, experts, gpu), torch.zeros_like(q8)
    sel2, weights2 = torch.zeros_like(sel), torch.zeros_like(weights)
    call("yvex_hip_moe_prepare_projecting", ptr(logits), None, u64(rows), u64(experts), u64(topk), C.c_int(K.SIGMOID), C.c_int(1),
         C.c_double(1.5), ptr(sel2), ptr(weights2), ptr(wl2.order), ptr(wl2.expert_ids), ptr(wl2.bucket_offsets),
         ptr(wl2.bucket_populations), ptr(wl2.sweep_offsets), ptr(wl2.counts), ptr(x), u64(hidden), u64(hidden), ptr(q82),
         C.byref(pair), ptr(status))
    assert torch.equal(sel2, sel) and same_bits(weights2, weights) and torch.equal(q82, q8)
    assert torch.equal(wl2.order, wl.order) and torch.equal(wl2.counts, wl.counts)
    assert same_bits(got[0], want[0]) and same_bits(got[1], want[1])
    assert lib.yvex_hip_q8k_quantize_swiglu_projecting_supported(ptr(down), u64(hidden), u64(middle // 32 * 34), u64(rows), u64(middle))
    mid2, got_down = torch.zeros_like(mid[0]), torch.full((rows, hidden), 7.0, device=gpu)
    call("yvex_hip_q8k_quantize_swiglu_projecting", ptr(routed), u64(rows * topk), u64(middle), ptr(mid2), ptr(want[0]),
         ptr(want[1]), u64(rows), C.c_double(limit), ptr(down), u64(hidden), u64(middle // 32 * 34), ptr(got_down), ptr(status))
    assert torch.equal(mid2, mid[0]) and same_bits(got_down, want_down)
    assert int(status.item()) == 0
    # three rows and matrices on odd addresses are refused
    assert not lib.yvex_hip_moe_prepare_projecting_supported(C.byref(pair), u64(3), u64(hidden))
    pair.second += 1
    assert not lib.yvex_hip_moe_prepare_projecting_supported(C.byref(pair), u64(rows), u64(hidden))
    assert not lib.yvex_hip_q8k_quantize_swiglu_projecting_supported(C.c_void_p(down.data_ptr() + 1), u64(hidden),
                                                                     u64(middle // 32 * 34), u64(rows), u64(middle))


# two workgroups a row (as many rows as the device leaves two compute units each) against one: the row in registers, rows too
# long for them, a width that is no multiple of four, other numbers of streams
@pytest.mark.parametrize("streams,width", [(4, 4096), (4, 7168), (4, 8448), (4, 510), (2, 256), (3, 4100), (7, 1024)])
def test_ingress_of_few_rows_is_that_of_many(gpu, oracle, streams, width):
    """A row's results do not depend on its batch."""
    from yvex_amd import kernels as K
    units = torch.cuda.get_device_properties(gpu).multi_processor_count
    g, count, mixing = oracle.Generator(42, f"ingress.{streams}.{width}"), units // 2 + 1, (streams + 2) * streams
    rows, mixes = (dev(g.normal(count * n).reshape(count, n), gpu) for n in (streams * width, mixing))
    scale, base, norm = (dev(g.normal(n), gpu) for n in (3, mixing, width))
    kw = dict(streams=streams, width=width, iterations=20, rms_epsilon=1e-6, mhc_epsilon=1e-6, post_multiplier=2.0)
    status = K.new_status(gpu)
    many = K.mhc_ingress(rows, mixes, scale, base, norm, status=status, **kw)
    for few in (1, units // 2):
        got = K.mhc_ingress(rows[:few].contiguous(), mixes[:few].contiguous(), scale, base, norm, status=status, **kw)
        assert all(same_bits(a, b[:few]) for a, b in zip(got, many))
    assert int(status.item()) == 0
    rows[0, streams * width - 1] = float("inf")
    K.mhc_ingress(rows[:1].contiguous(), mixes[:1].contiguous(), scale, base, norm, status=status, **kw)
    assert int(status.item()) == 1


# one and two workgroups a row, 256 and 1024 threads, 16- and 32-row tiles of the projection, two to 56 splits, one to four
# partial sums a thread; rows that fit LDS beside their collapsed values and not beside the partial sums as well; the widest row
@pytest.mark.parametrize("streams,width,count", [(2, 512, 8), (4, 1024, 20), (4, 1920, 300), (4, 4096, 8), (4, 4096, 96), (4, 4096, 129),
                                                 (4, 4096, 333), (7, 1024, 33), (7, 4096, 16), (7, 4096, 130), (4, 11520, 16),
                                                 (4, 12288, 8), (4, 12288, 96), (3, 14592, 8), (7, 16384, 8)])
def test_ingress_that_joins_its_projection_equals_the_launches_apart(gpu, oracle, streams, width, count):
    from yvex_amd import kernels as K, load_library
    g, mixing, expanded = oracle.Generator(46, f"projecting.{streams}.{width}"), (streams + 2) * streams, streams * width
    rows, function = dev(g.normal(count * expanded).reshape(count, expanded), gpu), dev(g.normal(mixing * expanded).reshape(mixing, expanded), gpu)
    function /= expanded ** 0.5
    scale, base, norm = (dev(g.normal(n), gpu) for n in (3, mixing, width))
    lib, status = load_library(), K.new_status(gpu)
    lib.yvex_hip_matvec_f32_scratch_bytes.restype = C.c_uint64
    need = lib.yvex_hip_matvec_f32_scratch_bytes(u64(mixing), u64(expanded), u64(count))
    scratch = torch.zeros(need // 8, dtype=torch.float64, device=gpu)
    kw = dict(streams=streams, width=width, iterations=20, rms_epsilon=1e-6, mhc_epsilon=1e-6, post_multiplier=2.0)

    def projecting(n):
        out = [torch.zeros(n, w, device=gpu) for w in (width, streams, streams * streams)]
        rc = lib.yvex_hip_mhc_ingress_projecting(
            ptr(rows), ptr(function), ptr(scale), C.c_uint(0), ptr(base), C.c_uint(0), ptr(norm), C.c_uint(0), u64(n), u64(streams),
            u64(width), u64(20), C.c_double(1e-6), C.c_double(1e-6), C.c_double(2.0), *(ptr(t) for t in out), ptr(scratch), u64(need),
            ptr(status), C.c_void_p(torch.cuda.current_stream().cuda_stream))
        return rc, out

    mixes = K.matvec_f32_rows(function, rows, status, scratch=scratch.view(torch.uint8))
    want = K.mhc_ingress(rows, mixes, scale, base, norm, status=status, **kw)
    rc, got = projecting(count)
    assert rc == 0 and int(status.item()) == 0
    assert all(same_bits(a, b.reshape(a.shape)) for a, b in zip(got, want))
    assert projecting(7)[0] != 0                   # a batch whose projection is one launch
    function[mixing - 1, 5] = float("inf")
    assert projecting(count)[0] == 0 and int(status.item()) == 1


def _row_with_mean_square_one(rng, width):
    """bf16 values, one of them 1.5, whose squares add up to `width` within 2^-70, most of them far below a unit in the
    last place of the large ones' squares: what a sum in double rounds to depends on its order."""
    row = np.exp2(rng.uniform(-22, -14, width)).astype(np.float32)
    row = (row.view(np.uint32) & 0xffff0000).view(np.float32)
    row[12] = 1.5
    left = (width << 80) - sum(int(float(v) * 2 ** 40) ** 2 for v in row[12:])
    for i in range(12):
        bits = np.float32((left / 2.0 ** 80) ** 0.5).view(np.uint32) & np.uint32(0xffff0000)
        if int(float(bits.view(np.float32)) * 2 ** 40) ** 2 > left:
            bits -= np.uint32(0x10000)
        row[i] = bits.view(np.float32)
        left -= int(float(row[i]) * 2 ** 40) ** 2
    assert 0 <= left < 1 << 10
    return rng.permutation(row)


# 256 and 1024 threads, a thread's columns the values that it adds and not, one and two columns a thread, longer rows
@pytest.mark.parametrize("width", [1024, 1536, 4096, 7168, 8704])
def test_ingress_adds_a_rows_squares_in_one_order(gpu, width):
    """Both sums of squares decide results: the one over the streams against a gate and a mixing logit from which all
    but its last places is taken away, the collapsed row's against a norm weight that puts 1.5 half way between
    two floats beside the middle of two bf16 values."""
    from yvex_amd import kernels as K
    streams, rng = 4, np.random.default_rng(width)
    units = torch.cuda.get_device_properties(gpu).multi_processor_count
    some = np.stack([np.concatenate([_row_with_mean_square_one(rng, width) for _ in range(streams)]) for _ in range(16)])
    count, mixing = units // 2 + 1, (streams + 2) * streams
    rows = dev(np.tile(some, (count // 16 + 1, 1))[:count], gpu)
    mix, base = np.zeros(mixing, np.float32), np.zeros(mixing, np.float32)
    base[:streams] = [100.0, -100.0, -100.0, -100.0]           # the first stream alone collapses
    for i in (streams, 2 * streams):                           # a post gate, a mixing logit
        mix[i], base[i] = 1.0, -2.0 ** 56
    mixes = dev(np.tile(mix, (count, 1)), gpu)
    scale = dev(np.array([0.0, 2.0 ** 56, 2.0 ** 56], np.float32), gpu)
    norm = torch.full((width,), 5614251.0 * 2.0 ** -23, device=gpu)
    kw = dict(streams=streams, width=width, iterations=1, rms_epsilon=2.0 ** -100, mhc_epsilon=2.0 ** -100, post_multiplier=2.0)
    status = K.new_status(gpu)
    many = K.mhc_ingress(rows, mixes, scale, dev(base, gpu), norm, status=status, **kw)
    for few in (1, units // 2):
        got = K.mhc_ingress(rows[:few].contiguous(), mixes[:few].contiguous(), scale, dev(base, gpu), norm, status=status, **kw)
        for a, b in zip(got, many):
            assert same_bits(a, b[:few])
    assert int(status.item()) == 0
