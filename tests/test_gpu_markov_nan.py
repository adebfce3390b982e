"""Draft selection over values that are all NaN: the argmax order of a NaN of all ones is 0, the order of no value at all,
and the row under it still has to be a row of the table (the first, as the keys' order says)."""
import numpy as np
import pytest

from conftest import load_host
from test_gpu_engine import SMALL, SMALL_WIDE, STOP_ANCHOR, make_weights, setup_caches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geom", [SMALL, SMALL_WIDE])
def test_every_value_a_nan_of_all_ones(geom):
    import torch
    host = load_host()
    desc = host.model_desc(**geom)
    print(f"case crop_rows={desc.crop_rows}", flush=True)
    eng = host.Engine(desc, 512)
    weights = make_weights(eng, desc, 11)
    eng.upload("markov.w2s", np.full(eng.tensor("markov.w2s")[1] // 4, 0xFFFFFFFF, np.uint32))
    a = 300
    setup_caches(eng, host, desc, a, 150, 111)
    eng.set_state(a=a, anchor=STOP_ANCHOR, count=0, rounds_left=1, limit=a + 40, budget=512, eos=-1, ctx_new=3,
                  ctx_pos=a - 3, ctx_lo=150, run=1, skip_rounds=1, stop_at=a + 64, ckpt_slot=-1, tokens=[STOP_ANCHOR])
    eng.round(0, a)
    torch.cuda.synchronize()
    keys = eng.download("keys", np.uint64, (2 * desc.block,))[desc.block:]
    state = eng.state()
    print("verified rows", state.M, "draft keys", [hex(k) for k in keys[:3]], flush=True)
    assert state.M >= 3
    assert list(state.tokens)[1:state.M] == [int(weights["crop_ids"][0])] * (state.M - 1)
    eng.close()
