// Configuration of the batched persistent solver per world-size bucket, from measurements on an MI355X
// with box2d_amd/autotune.py (which writes a file of this form with the fastest configuration of each
// bucket's batches alone). A batch's launch takes the size of the bucket with the most worlds; each world
// its bucket's warm-start form. The results do not depend on these values, only the time.
//
// Two sizes are not the tuner's, because a launch has one size and a batch's small worlds are the most but
// its large ones the longest: 256 threads for up to 64 bodies (alone 0.255 ms per step of 2,048 worlds,
// 128 threads 0.163; but 1,024 worlds of 8 to 1,024 bodies 0.371 against 0.621, 500 of 10 to 512 0.199
// against 0.288), and 512 for up to 1,024 (alone 0.240 ms per step of 256 worlds, 1,024 threads 0.201; but
// 200 worlds of 300 to 1,000 bodies and chains 0.236 against 0.255).
#pragma once

// { max awake bodies, workgroup threads, warm start body by body }
#define B2AMD_BATCH_TUNING_TABLE                                                                                         \
	{ { 64, 256, 0 }, { 256, 128, 0 }, { 1024, 512, 0 }, { 5400, 1024, 0 } }
#define B2AMD_BATCH_TUNING_SOURCE "box2d_amd/autotune.py, 2026-12-05; uneven batches"
