/*
 * varq_testing.h -- entry points of libvarq_hip.so that its tests need to reach and to recognise paths of varq_quant_pack, of the attention and of packing.  They are not part
 * of the interface and may change with any build; the conventions are those of varq.h.
 */
#ifndef VARQ_TESTING_H
#define VARQ_TESTING_H

#include "varq.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * varq_quant_pack with the time given that a workgroup waits for the others with which it shares its groups, in ticks of 10 ns, before
 * it helps to read their rows (0: without waiting).  Results do not depend on it.
 */
int varq_quant_pack_wait(const void *x, int x_dtype, const int64_t *host_shape4, int reduce_mask, int bits, int asym, float eps, int32_t *words,
                         int8_t *codes, float *scale, float *zp, const int64_t *host_out_map, uint32_t wait_ticks, void *workspace,
                         size_t workspace_bytes, void *stream);

/*
 * How varq_quant_pack (tensors = 1) or varq_quant_pack2 (2) go about a valid call on the current device: n > 1: that many workgroups share each
 * block of groups; 1: one workgroup takes each by itself; 0: neither, the input is read twice.  word_bits: bits of the packed codes, 8 for int8 codes.
 */
int varq_quant_pack_shards(const int64_t *host_shape4, int reduce_mask, int x_dtype, int tensors, int word_bits, int asym);

/*
 * Over how many wavefronts of a workgroup the attention shares the keys of its queries out on the current device when that is left to it (splits = 0) and
 * the kernel that widens per workgroup serves the call: 1, 2 or 4; 0: with these key limits K and V are expanded instead. nseg: tables (1 for scales per key); limits: whether there are key limits.
 */
int varq_fused_attn_key_waves(int B, int Hkv, int Lq, int Lk, int D, int nseg, int limits);

/*
 * varq_pack and varq_unpack with rows that do not fill their last word, or codes off 16 bytes, in launches of at most `stretch` codes each, padding included
 * (they count them in 32 bits).  by_pieces: 16 codes per thread (1, rows of 15 codes or more) or a word per thread (0).
 */
int varq_pack_stretches(const int8_t *codes, int64_t rows, int c, int bits, int32_t *words, int64_t stretch, void *stream);
int varq_unpack_stretches(const int32_t *words, int64_t rows, int c, int bits, int8_t *codes, int64_t stretch, int by_pieces, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* VARQ_TESTING_H */
