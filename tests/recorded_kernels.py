"""Which kernels a recording issues: the names in the library's own list of a recording's launches (HCHIP_RECORDING_LOG)."""


def kernels_of(backend, capfd, fn):
    """Records fn() and returns the names of the kernels in the recording (after the rewrite), in order."""
    capfd.readouterr()
    with backend.switches(HCHIP_RECORDING_LOG="1"):
        with backend.capture() as cap:
            kept = fn()
    cap.graph.destroy()
    del kept
    lines = [line for line in capfd.readouterr().err.splitlines() if line.startswith("hchip recording")]
    return [line.split(": ", 1)[1].split()[0] for line in lines]
