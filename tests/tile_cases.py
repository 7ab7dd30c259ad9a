"""Products that the rule on tile shapes (hy-mt-rs_amd/csrc/hyq_tile_pick.hpp)
sends to each shape, with a partial last token tile and, where the shape's row
count allows one, a partial last row tile."""

# (shape, weight rows, tokens) of a matmul at more than 128 tokens
MATMUL = [("T256", 14300, 777), ("T256R96", 12260, 300), ("T192", 14300, 300),
          ("T128", 6140, 600), ("T64", 200, 520)]
# (shape, gate rows, tokens) of a gate/up product (rows in whole 256s)
GATE_UP = [("T256", 7168, 777), ("T192", 7168, 300), ("T128", 3072, 600), ("T64", 1536, 500)]
