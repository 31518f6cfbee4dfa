"""Delta rule over chunks with the key channels shared by two waves: one and two groups of columns a workgroup, columns left over."""
import pytest
import torch

from docagents_amd.ops import get_ops
from seq_cases import Portions, close, rand
from test_zamitar import delta_case, delta_want

pytestmark = pytest.mark.gpu


# 60 heads of 3 groups of 16 columns and fewer: a group a workgroup; 72 heads of 5: two
@pytest.mark.parametrize("H,G,K,V", [(20, 4, 128, 40), (20, 4, 64, 24), (24, 8, 128, 72), (24, 24, 64, 72)])
def test_delta_rule_in_halves(H, G, K, V):
    P = Portions("cuda", "bf16", lens=(150, 33, 70), cuts=((70, 64, 16), (33,), (32, 38)))
    scale, eps = K ** -0.5, 1e-3
    qkv, dec, beta, gate = delta_case(P, H, G, K, V, K, V)
    dec[0].view(-1, H, K)[:, 0, 0] = -200.0  # forgets within a token: blocks of two scales
    weight = 1 + 0.3 * rand(9, V)
    state, conv = P.state(H, V, K), P.state(0, 2 * G * K + H * V, dtype=P.act)
    want = [delta_want(P.stored(qkv)[i], dec[i], P.stored(beta)[i], P.stored(gate)[i], H, G, K, V, K, V, weight, eps, scale)
            for i in range(3)]
    for m, spans in P:
        x = P.pack(qkv, spans)
        d = torch.cat([dec[i][a:b] for i, a, b in spans]).cuda().contiguous()
        got = get_ops("cuda").delta_rule(x, d, P.pack(beta, spans), state, x, conv, m, H, G, scale, 1e-6,
                                         (weight.cuda(), P.pack(gate, spans), V, eps)).view(m.T, H, V)
        row = 0
        for i, a, b in spans:
            close(got[row:row + b - a], want[i][0][a:b], "bf16")
            row += b - a
    for i in range(3):
        close(state[P.slots[i]].transpose(1, 2), want[i][1], "fp32", 2)
