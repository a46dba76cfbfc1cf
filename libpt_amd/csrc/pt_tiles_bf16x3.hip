/* Tile kernels of form PT_FORM_BF16X3 (pt_tiles.h). */
#include "pt_tiles.h"

extern "C" int
pt_launch_tiles_bf16x3(const struct pt_launch *p, int n, void *stream)
{
	return launch_form<PT_FORM_BF16X3>(p, n, (hipStream_t)stream);
}
