"""GPU: ptmi_model_generate's prompt pass (all forced positions at once)
against the oracle's token-by-token run (pt_text.c:344-350).

The last position's logits attend to every cached key and value, so they
check the caches of all prompt positions; one more forward_step checks that
the model goes on from them.  Tolerance: that of the decode step against the
oracle (1e-5 of max |logit|; only the orders of the sums differ).
"""
import numpy as np
import pytest

import pitorch_amd as pa
from tests._oracle import OracleModel

pytestmark = pytest.mark.gpu

SMALL = (64, 160, 2, 4, 4, 512, 256)             # dim hidden layers heads kv_heads vocab seq_len
PADDED_HEAD = (108, 260, 2, 3, 3, 512, 160)      # head_dim 36: no multiple of 16
WIDE_HEAD = (256, 512, 2, 2, 2, 512, 96)         # head_dim 128
ONE_LAYER = (96, 256, 1, 3, 3, 512, 96)          # keys and values only
WIDE = (2304, 260, 1, 24, 24, 512, 48)           # norm rows past one wave's registers
SPLIT_TILES = (768, 1280, 2, 12, 12, 512, 640)   # its long prompts' GEMMs run on the bf16-product tiles
TWO_PASSES = (32, 64, 2, 2, 2, 512, 1200)        # more positions than one pass takes


def test_long_prompts_take_the_split_tiles():
    D, H = SPLIT_TILES[:2]
    for n in (601, 617):
        for N, K, epi in ((3 * D, D, 1), (2 * D, D, 1), (2 * H, D, 2), (D, D, 0), (D, H, 0)):
            assert pa.gemm_plan(2, n, N, K, epilogue=epi, accumulate=not epi)[:3] == (64, 64, 0), (n, N, K)


@pytest.mark.parametrize("cfg,n_prompt,total", [
    *[(SMALL, n, n + 3) for n in (1, 2, 3, 4, 5, 6, 7, 9, 16, 17, 18, 33, 34, 65, 130, 253)],
    (SMALL, 40, 40), (SMALL, 40, 25), (SMALL, 40, 4), (SMALL, 40, 1), (SMALL, 256, 256),
    *[(PADDED_HEAD, n, n + 2) for n in (6, 31, 150)],
    *[(WIDE_HEAD, n, n + 2) for n in (6, 50, 90)],
    *[(ONE_LAYER, n, n + 2) for n in (6, 70)],
    *[(WIDE, n, n + 2) for n in (6, 40)],
    *[(SPLIT_TILES, n, n + 2) for n in (602, 618)],
    *[(TWO_PASSES, n, n + 2) for n in (1024, 1025, 1026, 1031, 1190)],
])
def test_prompt_pass_matches_oracle(cfg, n_prompt, total):
    blob = pa.synth_model(cfg, 21)
    prompt = np.array(pa.seed_tokens(n_prompt, n_prompt, cfg[5]), np.int32)
    m, om = pa.Model(blob), OracleModel(blob.copy())
    got = m.generate(prompt, total, stop_on_eos=False)
    want, tok = [], int(prompt[0])
    for pos in range(total):
        nxt = om.forward_step(tok)
        tok = int(prompt[pos + 1]) if pos + 1 < n_prompt else nxt
        want.append(tok)
    assert list(got) == want and m.pos() == total
    for step in range(2):
        lg, ref = m.logits(), om.logits()
        assert np.max(np.abs(lg - ref)) <= 1e-5 * np.max(np.abs(ref)), step
        if step or total == cfg[6]:
            break
        assert m.forward_step(tok) == om.forward_step(tok)
    # a second prompt on the same model: nothing of the first is left
    again = m.generate(prompt[::-1].copy(), total, stop_on_eos=False)
    m2 = pa.Model(blob)
    assert list(m2.generate(prompt[::-1].copy(), total, stop_on_eos=False)) == list(again)
    assert np.array_equal(m.logits(), m2.logits())
    m2.close()
    m.close()
    om.close()


def device_bytes_free():
    import ctypes
    from pitorch_amd._hip import hip
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_training_model_reserves_the_buffers_with_its_first_prompt():
    """A model that trains holds the prompt pass's buffers (here 8 Mi floats of
    split-K sums and 1024 rows) only once a prompt needs them."""
    cfg = (256, 512, 1, 4, 4, 512, 1024)
    blob = pa.synth_model(cfg, 23)
    m, m2 = pa.Model(blob, max_T=16), pa.Model(blob)
    prompt = np.array(pa.seed_tokens(4, 40, cfg[5]), np.int32)
    m.generate(prompt[:4], 8, stop_on_eos=False)
    before = device_bytes_free()
    got = m.generate(prompt, 48, stop_on_eos=False)
    held = before - device_bytes_free()
    assert held >= 4 * ((8 << 20) + 1024 * (6 * 256 + 512)) // 2
    assert list(got) == list(m2.generate(prompt, 48, stop_on_eos=False)) and np.array_equal(m.logits(), m2.logits())
    before = device_bytes_free()
    m2.generate(prompt, 48, stop_on_eos=False)
    m.generate(prompt, 48, stop_on_eos=False)
    assert before == device_bytes_free()
    m.close()
    m2.close()
