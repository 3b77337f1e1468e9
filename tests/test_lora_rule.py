"""Which of a LoRA term's products the fused kernels take from the library, on the CPU: the faster one at
measured sizes (microseconds of the library's products with the dropout kernels around them / of the
fused kernel on an MI355X, fp16, launches back to back)."""

import pytest

from solution.body import lora as L

# rule, (rows, width, rank, ...), library, fused
MEASURED = [
    (L._down_pays, (1000, 1536, 16, False), 4.9, 4.8),
    (L._down_pays, (2000, 512, 64, False), 5.6, 4.9),
    (L._down_pays, (5933, 1536, 16, False), 5.8, 7.6),
    (L._down_pays, (200, 8960, 64, False), 9.9, 40.4),
    (L._down_pays, (2000, 3584, 16, False), 6.2, 8.4),
    (L._down_pays, (5933, 1536, 16, True), 26.4, 12.0),
    (L._down_pays, (5933, 3584, 32, True), 32.2, 28.1),
    (L._down_pays, (2000, 896, 64, True), 14.8, 7.6),
    (L._down_pays, (64, 8960, 64, True), 20.9, 41.5),
    (L._down_pays, (40000, 896, 64, True), 48.1, 60.8),
    (L._dxa_pays, (5933, 1536, 16), 8.7, 6.1),
    (L._dxa_pays, (1000, 3584, 16), 9.6, 7.3),
    (L._dxa_pays, (2000, 8960, 32), 20.7, 33.8),
    (L._dxa_pays, (9000, 1536, 64), 13.8, 19.7),
    (L._down_grads_pay, (5933, 1536, 16, False, True), 29.1, 21.0),
    (L._down_grads_pay, (200, 3584, 64, False, True), 10.9, 15.6),
    (L._down_grads_pay, (9000, 8960, 64, False, True), 111.2, 144.5),
    (L._down_grads_pay, (5933, 1536, 16, True, True), 54.6, 26.2),
    (L._down_grads_pay, (200, 896, 64, True, True), 15.1, 20.3),
    (L._down_grads_pay, (4096, 1536, 16, False, False), 10.7, 15.0),
    (L._down_grads_pay, (9000, 1536, 16, False, False), 24.5, 17.8),
    (L._up_grads_pay, (5933, 1536, 16), 19.3, 14.9),
    (L._up_grads_pay, (4096, 8960, 16), 20.7, 26.7),
    (L._up_grads_pay, (64, 3584, 64), 6.8, 8.3),
    (L._base_pays, (16,), 10.9, 7.5),
    (L._base_pays, (64,), 12.9, 21.7),
]


@pytest.mark.parametrize("rule,args,library,fused", MEASURED)
def test_the_faster_one_is_taken(rule, args, library, fused):
    assert bool(rule(*args)) == (fused < library)
