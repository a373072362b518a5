"""What the host side decides for a call (kernels, attention key splits, workspaces, held device blocks), without a GPU:
the program tests/clients/host_checks.cpp calls the library's own functions."""
import os
import subprocess

import pytest

import test_gpu_attention_rows
import test_gpu_f32_rows
import test_gpu_layer_rows
import test_gpu_mid_rows

PROGRAM = os.path.join(os.path.dirname(os.path.abspath(__file__)), "clients", "_build", "host_checks")


def checks(*arguments):
    if not os.path.exists(PROGRAM):
        import __graft_entry__
        __graft_entry__.build()
    run = subprocess.run([PROGRAM, *(str(int(a) if isinstance(a, bool) else a) for a in arguments)],
                         capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, (arguments, run.returncode, run.stderr)
    return run.stdout


def split(batch, heads, kv_heads, head_dim, kv_bf16, length, source, causal):
    splits, chunk = map(int, checks("split", batch, heads, kv_heads, head_dim, kv_bf16, length, source, causal).split())
    return splits, chunk


@pytest.mark.parametrize("batch,length", [(1, 0), (0, 0), (0, 1), (0, 3), (0, 7), (0, 200)])
@pytest.mark.parametrize("head_dim", [8, 32, 64, 128])
@pytest.mark.parametrize("source", [0, 100, 5000])
@pytest.mark.parametrize("causal", [False, True])
def test_an_empty_chunk_or_batch_has_a_split(batch, length, head_dim, source, causal):
    # the launch refuses it afterwards: the arithmetic before that must not divide by its zero work-groups
    for kv_bf16 in (False, True):
        splits, chunk = split(batch, 8, 2, head_dim, kv_bf16, length, source, causal)
        assert splits >= 0 and chunk >= 0


@pytest.mark.parametrize("entry,staged,by_64_rows", [("linear", 3, 5), ("swiglu", 6, 10), ("attention", 8, 12)])
def test_a_call_that_fits_only_without_its_workspace_goes_on_without(entry, staged, by_64_rows):
    """300 rows of 512: a staged projection is three launches (rows, product, key slices), one without it five of 64
    rows; the attention module adds the fill of its cache's length and the attention itself."""
    assert int(checks("workspace", entry, 300, 512, -1)) == staged
    for left in (0, 1 << 16, 300 * 512 * 4):
        assert int(checks("workspace", entry, 300, 512, left)) == by_64_rows


@pytest.mark.parametrize("entry", ["linear", "swiglu", "attention"])
def test_no_staged_copy_past_4_gib_of_rows(entry):
    # the buffers are reserved, not touched
    few, many = (int(checks("workspace", entry, rows, 4096, -1)) for rows in (1 << 18, (1 << 18) + 1))
    assert few < 20 and many >= (1 << 18) // 64


def test_a_block_of_a_captured_graph_is_not_handed_out_again():
    # it belongs to the graph's allocation node: a free returns it to the runtime, also after the capture has ended
    returned, reused = map(int, checks("capture").split())
    assert returned == 1 and not reused


def test_held_blocks_are_not_freed_into_a_capture():
    # a free during a capture becomes a node of the graph, and each replay would free the block again
    assert checks("capture_release").split() == ["0", "0", "1"]


def test_the_peak_keeps_what_others_had_of_the_pool():
    alive, held, reset = (tuple(map(int, line.split())) for line in checks("peak").splitlines())
    assert alive == (4, 68)
    assert held[0] == 0 and 64 <= held[1] <= 68  # at most the held blocks too little
    assert reset == (0, 0)


@pytest.mark.parametrize("head_dim,length,source,split_up", [
    (2, 64, 256, False), (2, 32, 4096, False), (2, 16, 1024, False), (4, 64, 4096, False), (8, 64, 1024, False),
    (8, 32, 1024, False), (2, 4, 4096, True), (2, 8, 16384, True), (8, 8, 4096, True), (8, 4, 1024, True)])
def test_many_rows_of_small_heads_are_not_split(head_dim, length, source, split_up):
    # 4 sequences, 32 / 8 heads: a wave per query row, so many rows fill the device without key splits and their merge
    splits, chunk = split(4, 32, 8, head_dim, False, length, source, False)
    assert (splits > 1) == split_up and splits * chunk >= source


def test_freed_blocks_are_held_up_to_the_release_threshold():
    # held; at threshold 0 the held one goes back at once and a freed one is not held; held again
    assert checks("threshold").split() == ["1", "0", "0", "1"]


def test_an_allocation_that_fails_is_tried_again_without_the_held_blocks():
    assert checks("retry").split() == ["1", "1"]


# ------------------------------------------------------------------------------------------ kernels of the GPU tests
def projection(epilogue, rows, k, segments, bf16, bias=False, layer=False):
    return checks("projection", epilogue, rows, k, *(list(segments) + [0, 0])[:3], bf16, bias, layer).strip()


def layer_kernels(rows, d, heads, kv, hidden, bf16):
    side = kv * d // heads
    return [projection("qkv", rows, d, (d, side, side), bf16, layer=True),
            projection("residual", rows, d, (d,), bf16, layer=True),
            projection("swiglu", rows, d, (hidden, hidden), bf16, layer=True),
            projection("residual", rows, hidden, (d,), bf16, layer=True)]


def test_the_linear_tests_take_the_kernels_they_name():
    for rows, k, n, bias, kernel in test_gpu_mid_rows.LINEAR:
        assert projection("store", rows, k, (n,), True, bias) == kernel, (rows, k, n)
    for rows, k, n, shape in test_gpu_f32_rows.LINEAR_F32:
        assert projection("store", rows, k, (n,), False) == "f32 " + shape, (rows, k, n)
    for rows, k, n, shape in test_gpu_f32_rows.LINEAR_BF16:
        assert projection("store", rows, k, (n,), True) == "f32 " + shape, (rows, k, n)
    named = {kernel for *_, kernel in test_gpu_mid_rows.LINEAR}
    shapes = [{shape for *_, shape in table} for table in (test_gpu_f32_rows.LINEAR_F32, test_gpu_f32_rows.LINEAR_BF16)]
    assert named == {"mid", "narrow", "tiles"} and shapes == [{"32x16", "64x32", "64x64", "128x128"}] * 2


def test_the_layer_and_block_tests_take_the_kernels_they_name():
    for batch, length, d, heads, kv, hidden, rank, dtype, kernels, _ in test_gpu_layer_rows.LAYERS:
        assert layer_kernels(batch * length, d, heads, kv, hidden, dtype == "bf16") == kernels.split(", ")
        if rank == 16:
            assert projection("store", batch * length, d, (rank, rank), dtype == "bf16", layer=True) == "narrow"
    for batch, length, d, heads, kv, hidden, rank, _, kernels in test_gpu_mid_rows.PROMPTS:
        got = layer_kernels(batch * length, d, heads, kv, hidden, True)
        assert [kernel.split()[0] for kernel in got] == kernels.split(", "), (batch, length, d, hidden)
    for rows, hidden, kernels in test_gpu_mid_rows.SWIGLU:
        got = [projection("swiglu", rows, 512, (hidden, hidden), True), projection("store", rows, hidden, (512,), True)]
        assert [kernel.split()[0] for kernel in got] == kernels.split(", "), (rows, hidden)


def test_the_attention_tests_take_the_kernel_they_name():
    for B, H, KV, L, S, D, kernel in test_gpu_attention_rows.MANY:
        for bf16 in (False, True):
            for masked in (False, True):
                assert checks("attention", B, H, KV, D, bf16, L, S, False, masked).strip() == kernel


def test_the_prefill_parity_tests_take_the_kernels_they_name():
    assert layer_kernels(2 * 2048, 1024, 16, 4, 2816, True) == ["mid", "mid", "tiles", "mid"]
    assert layer_kernels(2 * 1024, 1024, 16, 4, 2816, True) == ["mid", "mid", "tiles", "mid"]
    assert layer_kernels(2 * 548, 1024, 16, 4, 2816, True) == ["mid"] * 4
    assert layer_kernels(4 * 2048, 512, 8, 2, 1536, True) == ["mid", "mid", "tiles", "mid"]
    assert layer_kernels(2 * 512, 256, 8, 2, 512, True) == ["mid"] * 4
    assert layer_kernels(4 * 4096, 2048, 32, 8, 5632, True) == ["tiles"] * 4
