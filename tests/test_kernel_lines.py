"""Which kernel a layer call is given on either side of the lines between the families that depend on the weight bytes of a
launch."""

import pytest


@pytest.mark.parametrize(
    "tokens,k,E,H,I,gate_up",
    [
        # 3.8 and 7.5 GB of weights per launch: streaming while an expert can hold at most 8 rows (where the narrow tiles are
        # 2 % faster: the row says where the line is, not where it belongs), narrow tiles up to 10 rows per expert, deep ones up to 80
        (8, 8, 256, 7168, 2048, "stream"),
        (9, 8, 256, 7168, 2048, "narrow"),
        (32, 8, 256, 7168, 2048, "narrow"),
        (320, 8, 256, 7168, 2048, "narrow"),
        (321, 8, 256, 7168, 2048, "tile_deep"),
        (2560, 8, 256, 7168, 2048, "tile_deep"),
        (2561, 8, 256, 7168, 2048, "tile_wide"),
        # a reduction of no whole 128 bytes is for the streaming kernel alone, as before
        (9, 8, 256, 7168 + 64, 2048, "stream"),
        # 0.7 and 1.5 GB: 20 and 104 rows per expert (streaming at 16 tokens, where the narrow tiles are up to 6 % faster: as above)
        (16, 8, 128, 4096, 1408, "stream"),
        (17, 8, 128, 4096, 1408, "narrow"),
        (320, 8, 128, 4096, 1408, "narrow"),
        (321, 8, 128, 4096, 1408, "tile_deep"),
        (1664, 8, 128, 4096, 1408, "tile_deep"),
        (1665, 8, 128, 4096, 1408, "tile_wide"),
        # 512 MiB, 576 MiB and 608 MiB: 28; from 640 MiB on 20
        (224, 8, 64, 4096, 1024, "narrow"),
        (225, 8, 64, 4096, 1024, "tile_deep"),
        (336, 8, 96, 3072, 1024, "narrow"),
        (337, 8, 96, 3072, 1024, "tile_deep"),
        (224, 8, 64, 4096, 1216, "narrow"),
        (160, 8, 64, 4096, 1280, "narrow"),
        (161, 8, 64, 4096, 1280, "tile_deep"),
        # 0.2 and 0.4 GB: 40 and 104
        (640, 8, 128, 2048, 768, "narrow"),
        (641, 8, 128, 2048, 768, "tile_deep"),
        (1664, 8, 128, 2048, 768, "tile_deep"),
        (1665, 8, 128, 2048, 768, "tile_wide"),
    ],
)
def test_lines_between_the_families(pra, tokens, k, E, H, I, gate_up):
    assert pra.layer_plan(tokens, k, E, H, I)["gate_up"] == gate_up
