"""device_to_host: the whole tableau as int32 entries, made on the host from
packed shots.  Sizes: the edges of a 64-column word and of a 64-shot group, and
enough shots that the packed shots come in several copies, cut inside a group."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B", [(1, 1), (1, 65), (7, 64), (31, 63), (32, 130), (63, 64),
                                 (64, 2500), (65, 70), (128, 1200), (300, 129)])
def test_entries_are_the_planes_bits(n, B):
    import plaquette_simulator as ps
    import plaquette_simulator_bindings as b
    from plaquette_simulator import workloads as W
    if b.device_count() < 1:
        pytest.skip("no GPU")
    st = ps.CliffordState(n, B, 5, True)
    ops = W.OpList()
    rng = np.random.default_rng(n + B)
    for _ in range(6 * n):
        q = int(rng.integers(0, n))
        ops.gate(int(rng.choice([W.OP_H, W.OP_S])), q)
        ops.with_prob(W.OP_H, q, 0.5)
        if n > 1:
            ops.with_prob(W.OP_CX, q, 0.5, (q + 1) % n)
        ops.noise(q, 0.2, 0.1, 0.2)
    st.run_program(ops.array(), "persistent")
    planes = np.asarray(st.read_planes(), np.uint64)  # [group][column][row]
    bits = np.unpackbits(planes.view(np.uint8).reshape(*planes.shape, 8), axis=-1,
                         bitorder="little")
    want = bits.transpose(0, 3, 2, 1).reshape(-1, 2 * n + 1, 2 * n + 1)[:B]  # [shot][row][column]
    for _ in range(2):  # the second call has the buffers
        x, z, r = st.device_to_host_numpy()
        assert x.dtype == np.int32 and x.shape == (B, 2 * n + 1, n)
        assert np.array_equal(x, want[:, :, :n])
        assert np.array_equal(z, want[:, :, n:2 * n])
        assert np.array_equal(r, want[:, :, 2 * n])
