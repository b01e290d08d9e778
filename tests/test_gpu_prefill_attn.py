"""The prefill attention at the edges of its tiles (16 query rows, 32 cache
rows a step, four waves): a prompt's logits, in one prefill and in two (the
second on a filled cache), against the same ids through the decode steps."""
import numpy as np
import pytest

import hiplm
import hipmoe
from common import model_case, rel_l2
from test_gpu_model import TIGHT

pytestmark = pytest.mark.gpu


# the second model's sliding window of 200 rows masks inside its longer prompts
@pytest.mark.parametrize("name,lengths", (("olmoe_prompt", (2, 15, 16, 17, 33, 129)),
                                          ("mixtral_window_prompt", (31, 130, 217, 239))))
def test_gpu_prefill_attention_tiles_vs_decode(name, lengths):
    md, prompt, case, _ = model_case(name)
    M = hiplm.LmModel(md, case[7])
    try:
        M.set_moe_path(hipmoe.PATH_GEMV)
        ids = np.resize(prompt, max(lengths))
        steps = [M.decode(int(i))[1].copy() for i in ids]
        for n in lengths:
            M.reset()
            whole = M.prefill(ids[:n])[1].copy()
            M.reset()
            M.prefill(ids[:n // 2])
            parts = M.prefill(ids[n // 2:n])[1]
            errs = rel_l2(whole, steps[n - 1]), rel_l2(parts, steps[n - 1])
            print(f"prefill attention {name} n={n}: {errs[0]:.2e} {errs[1]:.2e}", flush=True)
            assert max(errs) <= TIGHT
    finally:
        M.free()
