"""check_capacity's words, gathered 32 workspaces to a launch: every one of them is seen, whatever its place, and so are the append's bits and the largest escape count."""
import pytest
import torch

from gpu_util import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_ws", [0, 1, 31, 32, 33, 70])
def test_every_word_is_seen(n_ws):
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    from gaac_amd.kernel import AttnWorkspace
    cache = CompressedKVCache(300, 2, 64, device=dev)      # 600 heads: some threads look at none
    for i in range(n_ws): cache._partials[i] = AttnWorkspace(2, 2, torch.bfloat16, dev, with_out=False)
    cache.check_capacity()
    cache.check_capacity(used=5)
    for i in {0, 30, 31, 32, 63, 64, n_ws - 1} & set(range(n_ws)):
        cache._partials[i].epoch[1] = 1
        for kw in ({}, {"used": 5}):
            with pytest.raises(RuntimeError, match="re-arm"): cache.check_capacity(**kw)
        cache._partials[i].reset()
    for bits in (1, 2, 3):
        cache.overflow.fill_(bits)
        with pytest.raises(RuntimeError, match="lost data"): cache.check_capacity()
    cache.overflow.zero_()
    for st, h in ((cache.k, 0), (cache.v, 599), (cache.k, 64), (cache.v, 63)):
        cap = st.ovf_cap
        st.ovf_used[h] = cap - 1288      # one worst-case tile and the readers' padding fit: no more
        cache.check_capacity()
        assert cache.k.ovf_cap == cache.v.ovf_cap == cap
        st.ovf_used[h] += 1
        cache.check_capacity()
        assert cache.k.ovf_cap == cache.v.ovf_cap > cap
        st.ovf_used[h] = 0
