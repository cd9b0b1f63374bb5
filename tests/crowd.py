"""A lattice whose steps drive other lattices' DDFs from the last-level cache, so that their next
single step takes the launch for DDFs from HBM (step_shape, fx_abi.hip): the kernels of
large lattices, on lattices small enough for the oracle."""


class Crowd:
    def __init__(self):
        import fluidx3d_amd as fx
        self.lbm = fx.LBM(256, 256, 128, 1.0 / 6.0, storage="FP16S")  # 304 MiB of DDFs
        self.lbm.initialize()

    def run(self, lbm, cached=False):
        """One step of the crowd, one of lbm; asserts the launch that lbm's took."""
        from fluidx3d_amd import _abi
        self.lbm.run(1)
        lbm.run(1)
        form = lbm.ctx.launches().step_form
        assert bool(form & _abi.FX_FORM_CACHED) == cached, form
        return form

    def close(self):
        self.lbm.close()
