"""Which MLP sizes of the group configuration take the launch that stores the SwiGLU product only (no kernel runs here): launches that
leave compute units idle keep the two outputs, whose tiles are smaller."""
import pytest

from flh_amd.quantized_model.decoder_layer import W4A4DecoderLayer


@pytest.mark.parametrize("hidden,inter,rows,product", [
    (4096, 11008, 64, False), (4096, 11008, 65, True), (4096, 14336, 65, True), (4096, 14336, 4096, True),
    (4096, 5632, 65, False), (4096, 5632, 128, False), (4096, 5632, 129, True), (2048, 5632, 100, False), (2048, 5632, 129, True),
    (2048, 4096, 160, False), (2048, 4096, 256, True), (2048, 8192, 64, False), (2048, 8192, 65, True), (4096, 7168, 65, True),
    (1024, 2816, 65, False), (1024, 2816, 160, False), (1024, 2816, 256, True), (1024, 3584, 129, True), (1024, 2816, 2048, True)])
def test_line(hidden, inter, rows, product):
    layer = W4A4DecoderLayer(hidden, hidden // 128, hidden // 128, inter, activation="group", device="meta")
    assert layer._swiglu_gemm_applies(rows) == product
    token = W4A4DecoderLayer(hidden, hidden // 128, hidden // 128, inter, activation="token", device="meta")
    assert token._swiglu_gemm_applies(rows) == (rows > 64)
