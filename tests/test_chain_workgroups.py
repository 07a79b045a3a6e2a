"""How many workgroups a chain of the chunkwise bf16 rule takes, forward and backward, by the number of chains: what the library
launches, against a runtime that only writes it down."""
import pytest

from tests.test_handover_streams import on_host   # noqa: F401 (a fixture)


# 256 compute units: halves of 128 chains fill them; two rounds of halves against one of chains, three against two, four against
# two, five against three
@pytest.mark.parametrize("chains,seq,forward,backward", [
    (128, 2048, 1, 1), (129, 2048, 2, 2), (256, 2048, 2, 2), (257, 2048, 2, 1), (384, 512, 2, 1), (384, 448, 2, 2), (300, 64, 2, 2),
    (385, 2048, 2, 2), (513, 2048, 2, 2), (640, 2048, 2, 2), (1000, 2048, 2, 2)])
@pytest.mark.parametrize("rule", ["titans", "delta"])
def test_workgroups_of_a_chain(on_host, rule, chains, seq, forward, backward):   # noqa: F811
    on_host(f"""
n = 2 if "{rule}" == "titans" else 1
lib.{rule}_chunkwise_forward_bf16_rocm(*[some] * (3 + n + 1 + n + n + 1), {seq}, 64, {chains}, 64)
lib.{rule}_chunkwise_backward_bf16_rocm(*[some] * (3 + n + 1 + n + 1 + 3 + n + 1 + n), {seq}, 64, {chains}, 64)
ran = [name for name, _ in launches()]
s = int(n == 2)
for kernel in (f"cw_chain_fwd_kernelILb{{s}}ELb0ELi{forward}E", f"cw_adjoint_chain_kernelILb{{s}}ELi{backward}E"):
    assert sum(kernel in name for name in ran) == 1, (kernel, ran)
""")
