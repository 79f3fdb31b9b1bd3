// Generated by prolix_amd/tune.py -- pair-kernel settings measured fastest on
// the 256-system batched mix (mean ms per captured step). None differs from its
// default in prx_pair_dev.h.
#pragma once
