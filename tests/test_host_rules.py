"""What the host side decides for a call (attention key splits), without a GPU: the program
tests/clients/host_checks.cpp calls the library's own functions."""
import os
import subprocess

import pytest

PROGRAM = os.path.join(os.path.dirname(os.path.abspath(__file__)), "clients", "_build", "host_checks")


def checks(*arguments):
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
