"""3-qubit dense blocks on 33 qubits (FP32 storage, 64 GiB): 2^30 vectors in
2^24 workgroups, more than one dispatch takes.  A basis state becomes a column
of the block, in either half of the vectors and at every kind of offset."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.timeout(300)
def test_three_qubit_block_on_33_qubits():
    import spinoza_amd as spz
    from spinoza_amd import Unitary
    n, m = 33, 3
    rng = np.random.default_rng(5)
    q, _ = np.linalg.qr(rng.normal(size=(8, 8)) + 1j * rng.normal(size=(8, 8)))
    u = Unitary.from_matrix(q)
    s = spz.State(n, "f32")
    for t, control in ((0, -1), (4, 32), (17, -1), (17, 2), (n - m, -1)):
        for index in (5 << t, (1 << n) - 1 - (3 << t), (1 << 32) + 12345, 1 << 31):
            print(f"case 33q block t={t} c={control} index={index}", flush=True)
            s.set_basis(index)
            if control < 0:
                spz.transform_u(s, u, t)
            else:
                spz.c_transform_u(s, u, control, t)
            col = (index >> t) & 7
            base = index & ~(7 << t)
            on = control < 0 or (index >> control) & 1
            for j in range(8):
                want = q[j, col] if on else float(j == col)
                re, im = s.download(base + (j << t), 1)
                assert re[0] == np.float32(want.real) and im[0] == np.float32(want.imag), (j, want)
            assert abs(s.norm() - 1.0) < 1e-6
