"""256-query and 128-query workgroups on both sides of their rules (csrc/query_tile.hpp) and the cut last rounds of the former:
the kernels and workgroups that a call launches, forward and backward against an fp32 reference, head by head."""
import pytest

from tests.test_gpu_start_order import check

F4, F8, W, K, Q4, QW = "fwd_kernel<{D}, 0, 4, 0, 1, false>", "fwd_kernel<{D}, 0, 8, 0, 1, false>", "fwd_wide_kernel<{D}>", "fwd_keyshare_kernel<{D}, 8, 0>", \
    "bwd_dq_kernel<{D}, 0, 4, 0, 1>", "bwd_dq_wide_kernel<{D}>"
F4G, Q4G = F4.replace("1, false", "2, false"), Q4.replace("0, 1>", "0, 2>")          # two groups of wavefronts share the keys

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,launched", [
    # nothing excluded: a last round on an eighth of the units, in 32-query workgroups or the whole call in 128-query ones
    (1, 72, 1024, 832, 128, False, None, ((W, 256), (K, 256), (Q4, 576))), (1, 72, 1024, 768, 128, False, None, ((F4, 576), (Q4, 576))),
    (1, 68, 1024, 832, 64, False, None, ((W, 256), (K, 128), (Q4, 544))), (1, 68, 1024, 768, 64, False, None, ((F4, 544), (Q4, 544))),
    # on half of them: cut into 128-query ones, or throughout
    (1, 180, 512, 2112, 128, False, None, ((W, 256), (F4G, 208), (Q4, 720))), (1, 180, 512, 2048, 128, False, None, ((F4, 720), (Q4, 720))),
    (1, 180, 512, 3136, 64, False, None, ((W, 256), (F4G, 208), (Q4, 720))), (1, 180, 512, 3072, 64, False, None, ((F4, 720), (Q4, 720))),
    # the last key tile cut
    (1, 112, 1024, 1011, 128, False, None, ((F8, 448), (Q4, 896))), (1, 112, 1024, 499, 128, False, None, ((F4, 896), (Q4, 896))),
    # whole rounds: 128-query dQ up to 1536 keys, 2048 at D = 64
    (1, 128, 1536, 1600, 128, False, None, ((W, 768), (QW, 768))), (1, 128, 1536, 1536, 128, False, None, ((W, 768), (Q4, 1536))), (1, 96, 2048, 2048, 64, False, None, ((W, 768), (Q4, 1536))), (1, 96, 2048, 2112, 64, False, None, ((W, 768), (QW, 768))),
    # causal: other lengths, one round, the second round full, long walks
    (1, 200, 512, 1088, 64, True, None, ((F4, 800), (QW, 400))), (1, 200, 512, 1088, 128, True, None, ((F8, 400), (QW, 400))),
    (1, 64, 1024, 1024, 128, True, None, ((F4, 512), (Q4, 512))), (1, 80, 1536, 1536, 128, True, None, ((F8, 480), (Q4, 960))), (2, 16, 4096, 4096, 128, True, None, ((F8, 512), (QW, 512))),
    (2, 16, 4096, 4096, 64, True, None, ((F4, 1024), (Q4, 1024))),
    # key lengths: from two rounds on
    (4, 16, 2048, 1088, 128, False, (1088, 777, 64, 1000), ((F8, 512), (QW, 512))), (4, 15, 2048, 1088, 64, False, (1088, 777, 64, 1000), None)])
def test_launched(B, H, Sq, Sk, D, causal, lens, launched):
    got = [(name, n) for name, n in check(B, H, Sq, Sk, D, causal, lens, False) if name.startswith(("fwd_", "bwd_dq_")) and "merge" not in name]
    if launched is not None:
        assert got == [(name.format(D=D), n) for name, n in launched], got
    else:
        assert not any("wide" in name or ", 8>" in name for name, _ in got), got
