"""The library's rule is asked once per shape, not once per launch."""

import torch

from flagsparse_amd import _lib, _matrix


def test_rule_is_asked_once(monkeypatch):
    lib, asked = _lib.load(), []

    class Counting:
        def fsp_spmm_shares_nonzeros(self, *args):
            asked.append(args)
            return lib.fsp_spmm_shares_nonzeros(*args)

    monkeypatch.setattr(_lib, "load", Counting)
    _matrix._shares_nonzeros.cache_clear()
    data, perm = torch.ones(100), torch.arange(100, dtype=torch.int32)
    for _ in range(3):
        assert _matrix._permuted_in_kernel(data, perm, 64, 500, 400, 64, 16)
        assert _matrix._permuted_in_kernel(data, perm, 64, 500, 400, 64, 16, True)
        assert not _matrix._permuted_in_kernel(data, perm, 64, 1 << 20, 400, 64, 16)
        assert not _matrix._permuted_in_kernel(data, perm.long(), 64, 500, 400, 64, 16)
    assert len(asked) == 3
    _matrix._shares_nonzeros.cache_clear()
