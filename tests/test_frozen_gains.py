"""A frozen fp32 RMSNorm gain is cast anew by every forward: a write through ``.data`` moves no version counter."""

import torch

from speculators_amd.weights import WeightStager


def test_a_write_through_data_is_seen_by_the_next_forward():
    st, p = WeightStager(), torch.nn.Parameter(torch.ones(64), requires_grad=False)
    with torch.autocast("cpu", torch.bfloat16):
        st.begin()
        assert (st.gain(p) == 1).all() and st.gain(p).dtype == torch.bfloat16
        p.data.fill_(3.0)
        st.begin()
        assert (st.gain(p) == 3).all()


def test_a_gain_that_trains_without_a_graph():
    st, p = WeightStager(), torch.nn.Parameter(torch.full((64,), 2.0))
    with torch.autocast("cpu", torch.bfloat16), torch.no_grad():
        st.begin()
        assert (st.gain(p) == 2).all() and not st.gain(p).requires_grad
