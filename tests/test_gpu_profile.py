"""The bytes that the per-pass timer reports are those of the launches it times."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("forced", (False, True))
@pytest.mark.parametrize("N", [(32, 32, 32), (64, 32, 32), (96, 32, 32)])
def test_xforward_bytes_count_the_kept_stage_field(N, forced):
    """A chained x-forward writes its stage output in stage 3 alone, where that is kept: N1 <= 32 and forced states."""
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context, Plan, State
    print(N, forced, flush=True)
    p = Plan(Context(0), N)
    s = State(p)
    s.upload([p.to_dev(torch.zeros(p.shape, dtype=torch.complex128).numpy()) for _ in range(3)])
    if forced:
        s.set_force(1, 1.5, 3.5, 0.3, 0.1)
    b = [s.profile_passes(1e-3, nu=1e-2, stage=k, nrep=1)[1][4] for k in (1, 2, 3, 4)]
    nkx, nky, nkz = 2 * (N[0] // 3) - 1, N[1] // 3 + N[1] - (2 * N[1] // 3 + 2), N[2] // 3
    state, lines = 16 * 3 * nkx * nky * nkz, 16 * (6 + 3) * N[0] * nky * nkz
    kept = forced or N[0] <= 32
    # stage 1: state read, accumulator written; 2 and 3: state and accumulator read, accumulator written; 4: state
    # and accumulator read, state written
    assert b == [lines + 2 * state, lines + 3 * state, lines + (4 if kept else 3) * state, lines + 3 * state]
