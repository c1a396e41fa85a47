"""Names of the reference's module that a caller may use beside the public ones."""
import oregon_gpt_oss_patching_amd.attention_kernel as ak


def test_the_autograd_function_goes_by_its_name():
    assert ak._attention.apply is ak.attention
