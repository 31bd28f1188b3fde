"""The phase clock is in every flash kernel of the instrumented library and in
none of the product: read from the AMD assembly of both, so no GPU is needed."""

import re

# clock reads per kernel: its start, the loop's start and end, its end, and the
# same two ends by the real-time clock; then the waits, score and output phases
LIFETIME, REAL_TIME, PHASES = 4, 2, 5


def _flash_kernels(asm):
    return {name: body for name, body in
            re.findall(r"^(_Z\w*(?:flash\w*|slice\w*)_kernel\w*):.*?\n(.*?)^\s*s_endpgm", asm,
                       re.S | re.M)}


def _kernels(device_asm, library):
    return {name: body for (_, lib), asm in device_asm.items() if lib == library
            for name, body in _flash_kernels(asm).items()}


def test_every_flash_kernel_is_stamped(device_asm):
    kernels = _kernels(device_asm, "kernels_phaseclock.so")
    assert len(kernels) == 6 + 12 + 2  # fp32 forms, 16-bit forms, the fp32 slice form
    for name, body in kernels.items():
        assert body.count("s_memtime") >= LIFETIME + PHASES, name
        assert body.count("s_memrealtime") >= REAL_TIME, name


def test_the_product_is_not(device_asm):
    kernels = _kernels(device_asm, "kernels.so")
    assert len(kernels) == 6 + 12 + 2
    assert not [name for name, body in kernels.items() if "s_memtime" in body]
