/*
 * Entry points of liba8attn.so for the streaming vocoder beyond the reference's operators (a8attn.h holds those).
 * Conventions (strides in elements, status codes, streams) are a8attn.h's.
 */
#ifndef A8VOC_H
#define A8VOC_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * a8_conv_cl_snake: a8_conv_cl whose stored outputs pass through a second snake, y <- y + out_ib sin(out_a y)^2 on the
 * fp16 outputs (fp32 arithmetic, rounded to fp16 again): the bits a conv with that snake on its loads would see. For a
 * conv whose output only feeds such a conv. out_a / out_ib fp32 [Cout], 16-byte aligned, or both NULL (then the call
 * is a8_conv_cl). No counterpart in the reference, whose conv_cl applies the snake on the next conv's loads
 * (serve/fast_engine.py:218-233). Workspace: a8_conv_cl_ws_bytes.
 */
int a8_conv_cl_snake(const void *x, int64_t s_xb, int64_t s_xt, const void *w, int64_t s_wp, int64_t s_wt,
                     int64_t s_wc, int cout_w, const void *bias, const void *res, int64_t s_rb, int64_t s_rt, void *y,
                     int64_t s_yb, int64_t s_yt, const float *snake_a, const float *snake_ib, const float *out_a,
                     const float *out_ib, int B, int Tin, int TR, int Cin, int Cout, int taps, int dil, int ph,
                     void *ws, int64_t ws_bytes, void *stream);

/*
 * a8_conv_tile_query: which instance of the tile kernel a8_conv_cl (ru = 0) or a8_ru_cl (ru = 1; Cin = Cout) takes for
 * contiguous, aligned operands of these sizes, without a snake on the loads, and a workspace of ws_bytes: *mt the 32-row
 * groups of a wave (2 or 3), *xkb the KiB of one slice of input rows, *ksplit the K shares; *mt = *xkb = 0 where the
 * call runs on the general kernel. Host arithmetic, nothing is launched. For tests and tuning.
 */
int a8_conv_tile_query(int B, int Tin, int TR, int Cin, int Cout, int taps, int dil, int ph, int ru, int64_t ws_bytes,
                       int *mt, int *xkb, int *ksplit);

#ifdef __cplusplus
}
#endif
#endif
