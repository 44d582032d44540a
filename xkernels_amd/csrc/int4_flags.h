// Bits of the int4 `flags` argument that are not part of the public ABI.
//
// The public value is 0 (include/xk_moe.h). The bits below pick a kernel where
// the shapes allow more than one, so the GPU tests can compare the prefill tile
// kernel with the decode stream kernel on the same inputs. Callers outside the
// tests leave them clear; any other bit is rejected.
#pragma once

#define XK_INT4_TEST_FORCE_TILE (1 << 8)
#define XK_INT4_TEST_FORCE_STREAM (1 << 9)
// with FORCE_TILE: the 256-row tile kernel where it takes the shape
#define XK_INT4_TEST_TALL (1 << 11)
#define XK_INT4_TEST_BITS (XK_INT4_TEST_FORCE_TILE | XK_INT4_TEST_FORCE_STREAM | XK_INT4_TEST_TALL)
// Set by the fused call (and the query of its kernel) alone, never accepted from
// a caller: K or N not a multiple of 256 may take the tile kernel. The stage
// entry keeps such shapes on the stream kernel, whose calls may come without
// align outputs and with the plane count it answers.
#define XK_INT4_FUSED (1 << 10)
