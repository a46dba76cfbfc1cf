/* Tile kernels of form PT_FORM_FP32 (pt_tiles.h). */
#include "pt_tiles.h"

extern "C" int
pt_launch_tiles_fp32(const struct pt_launch *p, int n, void *stream)
{
	return launch_form<PT_FORM_FP32>(p, n, (hipStream_t)stream);
}
