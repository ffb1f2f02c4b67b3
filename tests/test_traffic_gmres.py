"""The counter post-processing counts the (F)GMRES vector kernels with the BLAS class."""
from asam_amd import traffic


def test_gmres_kernel_classes():
    c = traffic.kernel_class
    assert c("void asam::k_gm_dot<double, true>(long, double const*, ...)") == "blas_fp64"
    assert c("void asam::k_gm_dot<float, false>(long, float const*, ...)") == "blas_fp32"
    assert c("void asam::k_mgs<double, 3, 3>(long, double*, asam::MgsVecs, ...)") == "blas_fp64"
    assert c("void asam::k_mgs<float, 1, 0>(long, float*, asam::MgsVecs, ...)") == "blas_fp32"
