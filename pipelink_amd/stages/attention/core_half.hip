// Package fa.core of half tiles: the whole tiles' source compiled for 64 queries a workgroup.  The same stage with the same
// seams, params and handles, so a pipeline.json takes either by its artifact_path.
#define FA_HALF_TILES 1
#include "core.hip"
