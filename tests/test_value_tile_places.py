"""The exchange between lanes in `store_value_tile` (common.hpp): what the lanes of the first wavefront tell each other about their tokens' places goes
from lane to lane.  Places that a lane has written to LDS are read by others behind the barrier alone."""
import os
import re

import llmserver_amd


def test_no_lane_reads_anothers_place_in_front_of_the_barrier():
    with open(os.path.join(os.path.dirname(llmserver_amd.__file__), "csrc", "common.hpp")) as handle:
        source = re.sub(r"//[^\n]*", "", handle.read())
    body = source[source.index("void store_value_tile("):]
    sorting = body[body.index("if (threadIdx.x < VT_TOKENS)"):body.index("__syncthreads();")]
    assert re.findall(r"place_of\[[^\]]*\][^;]*;", sorting) == ["place_of[t] = place;"]
