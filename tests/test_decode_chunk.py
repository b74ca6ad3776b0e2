"""What a workgroup of the decode kernel takes of a context (``ops.decode_chunk``), on either side of where whole contexts begin."""
import pytest

from glassbox_amd import ops


@pytest.mark.parametrize("n, kv_heads, head_dim, bucket, whole", [
    (1, 1, 64, 512, True), (1, 1, 128, 512, True),
    (16, 5, 64, 1024, True), (15, 5, 64, 1024, False), (48, 3, 64, 2048, True), (47, 3, 64, 2048, False),
    (18, 8, 128, 1024, True), (20, 8, 128, 1024, True), (17, 8, 128, 1024, False),
    (24, 8, 128, 2048, True), (23, 8, 128, 2048, False),
    (32, 8, 128, 4096, True), (31, 8, 128, 4096, False), (8, 32, 64, 8192, True), (7, 32, 64, 8192, False)])
def test_whole_contexts_where_there_are_workgroups_enough(n, kv_heads, head_dim, bucket, whole):
    chunk = ops.decode_chunk(n, kv_heads, bucket, head_dim)
    assert chunk % 256 == 0 and (chunk >= bucket) == whole
    assert -(-bucket // chunk) <= 256      # what the second pass combines
