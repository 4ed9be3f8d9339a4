"""What the batched form asks of the HIP runtime, on the stand-in of test_transfer_runtime."""
import pytest

from test_transfer_runtime import child  # noqa: F401 (fixture)


@pytest.mark.parametrize("first", ["fp64", "mixed"])
def test_persistent_grid_belongs_to_its_kernel(child, first):  # noqa: F811
    """The workgroups of the persistent schedule follow from the kernel and the workgroup it is launched
    with (the stand-in: four of 256 lanes a compute unit in FP64, of which twice as many are launched, five
    in FP32; 256 compute units), whichever precision or size of workgroup the process batched first."""
    child(f"""
def grid(precision, N, tile):
    members = [gpu.DGSEM(C.euler_vortex_case(60, N), precision) for _ in range(12)]
    b = gpu.Batch(members, tile, 4, use_graph=False)
    F.fake_watch(b"k_batch_stage_persist")
    b.rk_step(0.0, np.full(len(members), 1e-3))
    n = F.fake_grid()
    b.close()
    [m.close() for m in members]
    return n
order = [{first!r}] + [p for p in ("fp64", "mixed") if p != {first!r}]
got = {{p: grid(p, 8, 1) for p in order}}
assert got == {{"fp64": 2 * 4 * 256, "mixed": 5 * 256}}, got
# P = 5: workgroups of one wavefront in the narrow tile; P = 9: of two
assert [grid("fp64", N, 0) for N in (8, 4)] == [2 * 8 * 256, 2 * 16 * 256]
""")
