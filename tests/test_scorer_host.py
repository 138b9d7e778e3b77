"""CPU: what the scorers' host side hands to the library (workspaces, which calls it takes), no kernels run."""
import pytest


@pytest.mark.parametrize("batch,cols", [(1, 4096), (1, 3584), (2, 256), (7, 1024), (600, 64)])
def test_the_mean_of_a_prompt_without_its_sinks_fits_the_workspace_of_the_whole_prompt(batch, cols):
    # a prompt's workspace is asked for with all its tokens, the mean then leaves the sinks (up to 64 tokens) out
    from kvquant import _lib
    need = _lib.lib.odmkv_token_mean_workspace_bytes
    for rows in [*range(1, 700), *range(8100, 8500), 32768, 65537, 131072 + 4]:
        whole = need(batch, rows, cols)
        assert all(need(batch, rows - n, cols) <= whole for n in range(1, min(rows, 65)))


@pytest.mark.parametrize("batch,cols", [(1, 4096), (1, 3584), (2, 256), (7, 1024), (600, 64)])
def test_the_mean_workspace_holds_every_run_of_rows(batch, cols):
    # the kernel's cut: runs of 16 to 256 rows, as many as put two workgroups on each of 256 compute units
    from kvquant import _lib
    for per_thread in (8, 4):
        runs = max(1, 512 // (batch * -(-cols // (256 * per_thread))))
        for rows in (1, 15, 16, 17, 4095, 4097, 8189, 8193, 65537, 131073, 131072 * 2 + 1):
            chunk = min(256, max(16, -(-rows // runs)))
            assert _lib.lib.odmkv_token_mean_workspace_bytes(batch, rows, cols) >= batch * -(-rows // chunk) * cols * 4
