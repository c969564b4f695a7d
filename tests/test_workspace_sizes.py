"""Sizes that the C ABI asks scratch of: no more than a launch of the same sizes and type would use."""
from fastgl import _lib as L


def test_weight_grad():
    lib = L.lib()
    # beyond what is formed in parts, which would want eight times as much (k = 100 K, 4096 x 4096: 64 x 64 tiles of one sum each)
    assert lib.fgl_weight_grad_workspace_bytes(100_000, 4096, 4096) < 70 << 20
    for k, m, n in ((3000, 602, 4000), (8000, 602, 1000), (107_000, 100, 256), (1000, 1000, 1000), (5, 64, 64)):
        fp32, bf16 = (lib.fgl_weight_grad_workspace_bytes_for(k, m, n, d) for d in (L.F32, L.BF16))
        assert bf16 <= fp32 == lib.fgl_weight_grad_workspace_bytes(k, m, n)
    assert 4 * lib.fgl_weight_grad_workspace_bytes_for(3000, 602, 4000, L.BF16) < lib.fgl_weight_grad_workspace_bytes_for(3000, 602, 4000, L.F32)
