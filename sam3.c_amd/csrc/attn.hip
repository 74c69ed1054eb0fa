/*
 * attn.hip - fused scaled dot-product attention (flash-attention forward)
 * for gfx950: out = softmax(Q K^T / sqrt(D) + mask) V per head, without
 * materializing the [Sq, Sk] score matrix. Replaces cpu_kernel_sdpa
 * (src/backend/cpu/kernels/cpu_sdpa.c:216-288), whose per-row online
 * softmax (sdpa_row_f32, :49-159) this follows one 64-key tile at a time.
 *
 * Layout: Q [BH, Sq, D], K and V [BH, Sk, D], out [BH, Sq, D], all of one
 * dtype (f32, bf16 or f16); the optional additive mask is f32 [Sq, Sk],
 * shared by all heads (cpu_sdpa.c:193-196).
 *
 * attn_fwd (D = 64, 16-byte aligned tensors): a workgroup (4 waves) owns
 * 128 queries of one head; wave w owns 32. The scores are computed
 * transposed, S^T = K Q^T, with v_mfma_f32_32x32x16: a lane then holds one
 * query (lane & 31) and 32 of the tile's 64 keys, so the row max and row
 * sum are in-lane reductions plus one exchange with lane ^ 32. The output
 * is accumulated transposed too, O^T = V^T P^T: the P^T operand is exactly
 * the lane's own probabilities (the MFMA's k index is permuted the same
 * way for both operands, which leaves the product unchanged), and the
 * per-query rescale exp(m_old - m_new) is a per-lane scalar.
 *   - bf16/f16: K tiles arrive in LDS by direct-to-LDS loads
 *     (XOR-swizzled rows); V tiles are staged through registers and
 *     written transposed, V^T [D][64 keys], row pitch 136 bytes;
 *   - f32: every operand is split into two bf16 planes, x = hi + lo with
 *     hi = bf16(x), lo = bf16(x - hi), and each product is formed as
 *     hi*hi + lo*hi + hi*lo (the dropped lo*lo term is below 2^-16 of the
 *     product), so f32 inputs keep about 16 significant bits per product at
 *     three bf16 MFMAs per tile step. K and V are split while they are
 *     staged into LDS through registers;
 *   - keys past Sk get a -inf score, queries past Sq are not stored;
 *   - scores are scaled into base 2 (exp2 = v_exp_f32).
 *
 * attn_generic: any D up to 512 and any element alignment, one wave per
 * query row, f32 arithmetic with expf: the path for the reference's other
 * head sizes (the mask decoder's 32, the prompt encoder's 16).
 */
#include "gemm_common.h"
#include "lds_dma.h"

namespace s3k {

struct AttnArgs {
	const char *q, *k, *v;
	const float *mask;
	char *out;
	int Sq, Sk;
	long long hq, hk;       /* per-head strides, elements */
	int BH, nqb;            /* heads, query blocks per head */
	int mask_vec;           /* mask rows 16-byte aligned: float4 loads */
	int oh;                 /* > 0: output head-merged (at_out_row)      */
	int ofmt;               /* merged f32 rows written as a GEMM operand:
				 * 0 f32, 1 bf16 planes [hi|lo] (row pitch
				 * 2*oh*D), 2 f16 with the range flag        */
	unsigned *ovf;          /* ofmt 2: range flag (or NULL) and its tag  */
	unsigned ovf_tag;
};

/* Element offset of output row q of head hh: [BH, Sq, D] rows, or with
 * oh > 0 heads merged, hh = b*oh + h stored as row b*Sq + q, columns
 * h*D.. of [B*Sq, oh*D] (the permute (0,2,1,3) of [B, oh, Sq, D]). */
__device__ __forceinline__ long long at_out_row(int oh, long long hh, int Sq, int q, int D)
{
	if (oh <= 0)
		return (hh * Sq + q) * (long long)D;
	const long long b = hh / oh, h = hh - b * oh;
	return ((b * Sq + q) * oh + h) * (long long)D;
}

constexpr int AT_D = 64, AT_BKV = 64;
constexpr int AT_VT_PITCH = AT_BKV * 2 + 8;          /* bytes per V^T row */
constexpr int AT_K_BYTES = AT_BKV * AT_D * 2;        /* 8 KiB per plane */
constexpr int AT_VT_BYTES = AT_D * AT_VT_PITCH;      /* 8.5 KiB per plane */

/* VD: V tiles by direct-to-LDS loads, row-major [key][d], read as the
 * V^T operand with transposing LDS reads (16-bit inputs); else staged
 * through registers into a V^T tile */
template <int DT, int NW, bool VD = false>
struct AtCfg {
	static constexpr bool SPLIT = DT == S3K_F32;
	static constexpr int NPL = SPLIT ? 2 : 1;        /* bf16 planes */
	static constexpr int KS = NPL * AT_K_BYTES;      /* one K slot */
	static constexpr int VS = VD ? AT_K_BYTES : NPL * AT_VT_BYTES; /* one V slot */
	static constexpr int LDS = 2 * KS + 2 * VS;      /* two of each */
	static constexpr int FAM = DT == S3K_F16 ? FAM_F16 : FAM_BF16;
	static constexpr int BQ = 32 * NW;                /* queries per workgroup */
	static constexpr int KJ = (8 + NW - 1) / NW;      /* K loads per wave */
};

template <int DT>
__device__ __forceinline__ uint32_t at_pack2(float lo, float hi)
{
	if constexpr (DT == S3K_F16)
		return pack_f16x2(lo, hi);
	else
		return pack_bf16x2(lo, hi);
}

/* f32 sum of the two 16-bit values of w, added to acc (v_dot2 with 1, 1) */
template <int DT>
__device__ __forceinline__ float at_sum2(uint32_t w, float acc)
{
	if constexpr (DT == S3K_F16) {
		typedef _Float16 h2 __attribute__((ext_vector_type(2)));
		const h2 one = {(_Float16)1.0f, (_Float16)1.0f};
		return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, w), one, acc, false);
	} else {
		const s3k_bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
		return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(s3k_bf16x2, w), one, acc, false);
	}
}

/* Chunk swizzle of a direct-to-LDS V tile row: it depends on the key's
 * low four bits only, so the transposed reads of the four 16-key chunks
 * of a tile differ by a constant offset. */
__device__ __forceinline__ int at_vswz(int key)
{
	const int r = key & 15;
	return (r ^ (r >> 3)) & 7;
}

typedef short at_v4i16 __attribute__((ext_vector_type(4)));

/* ds_read_b64_tr_b16: within each group of 16 lanes, lane i receives
 * element i % 4 of the 8 bytes addressed by lanes i / 4, 4 + i / 4,
 * 8 + i / 4 and 12 + i / 4 (measured on gfx950). */
__device__ __forceinline__ uint2 at_read_tr(const char *smem, unsigned off)
{
	const at_v4i16 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
		(__attribute__((address_space(3))) at_v4i16 *)((__attribute__((address_space(3))) char *)
								       smem + off));
	return __builtin_bit_cast(uint2, r);
}

/* x combined with the value of lane ^ 32 (v_permlane32_swap) */
__device__ __forceinline__ float at_max_pair(float x)
{
	const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
	return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float at_sum_pair(float x)
{
	const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
	return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

/* hi/lo bf16 planes of two f32 values, one dword each */
__device__ __forceinline__ void at_split2(float a, float b, uint32_t &hi, uint32_t &lo)
{
	hi = pack_bf16x2(a, b);
	lo = pack_bf16x2(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xFFFF0000u));
}

__device__ __forceinline__ void at_split8(const float4 &x, const float4 &y, uint4 &hi, uint4 &lo)
{
	at_split2(x.x, x.y, hi.x, lo.x);
	at_split2(x.z, x.w, hi.y, lo.y);
	at_split2(y.x, y.y, hi.z, lo.z);
	at_split2(y.z, y.w, hi.w, lo.w);
}

/* workgroups per CU the registers are budgeted for, chosen so that no
 * variant spills: three (12 waves, 168 VGPRs) for the 16-bit kernel
 * without a mask, two for f32 or a mask, one for f32 with a mask (its
 * mask tile, score halves and hi/lo operand planes need 256+ VGPRs) */
template <int DT, int NW, bool MASK, bool VD = false>
constexpr int at_minb()
{
	return NW != 4 ? 1 : (DT == S3K_F32 && MASK) ? 1 : (DT == S3K_F32 || MASK) ? 2 : 3;
}

template <int N>
struct at_int {
	static constexpr int value = N;
};

/* The probabilities of half a tile are formed against the running max m
 * without first taking the tile's max: they are only recomputed (after
 * moving m to the tile's max and rescaling the accumulators) when some
 * lane's 32 probabilities sum past 2^15, which also catches the first
 * tile (m = -FLT_MAX gives +inf). Every probability the MFMA sees is
 * then below 2^15, inside the f16 range. */
constexpr float AT_PSUM_MAX = 32768.0f;

/* The max m is moved to when half 0 of a tile is redone also covers half 1,
 * whose scores are then still without their mask and with zeros for keys
 * past Sk: m may pass the scores that count, by up to 2^AT_SLACK. All
 * probabilities then carry a factor down to 2^-AT_SLACK, which the division
 * by their sum takes out: exact in the exponent range of f32 and bf16; in
 * f16 it costs 8 of the 24 binary places between 1 and the smallest
 * subnormal. Past the slack (scores of -200 beside a key that does not
 * exist) it would turn them all into zeros: half 0 then takes its own max. */
template <int DT>
constexpr float AT_SLACK = DT == S3K_F16 ? 8.0f : 64.0f;

template <int DT>
__device__ __forceinline__ float at_new_max(float m_run, float own, float other, bool other_counts)
{
	constexpr float LOG2E = 1.44269504088896341f;
	const float mo = fmaxf(m_run, at_max_pair(own) * LOG2E);
	const float ma = fmaxf(mo, at_max_pair(other) * LOG2E);
	return !other_counts && ma - mo > AT_SLACK<DT> ? mo : ma;
}

/* Normalize (a query with no finite score keeps zeros, as the reference's
 * row_sum > 0 test leaves it) and store out[q][d] from a wave's O^T. */
template <int DT>
__device__ __forceinline__ void at_store(const AttnArgs &p, const s3k_f32x16 (&o)[2], float l_run,
					 long long head, int q, int h)
{
	const float l_tot = at_sum_pair(l_run);
	const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
	if (q < p.Sq) {
#pragma unroll
		for (int md = 0; md < 2; ++md)
#pragma unroll
			for (int g = 0; g < 4; ++g) {
				const int d0 = 32 * md + 8 * g + 4 * h;
				const float x0 = o[md][4 * g] * inv, x1 = o[md][4 * g + 1] * inv;
				const float x2 = o[md][4 * g + 2] * inv, x3 = o[md][4 * g + 3] * inv;
				const long long orow = at_out_row(p.oh, head, p.Sq, q, AT_D);
				if constexpr (DT == S3K_F32) {
					if (p.ofmt == 1) {
						/* the merged row r = orow / K as bf16 planes,
						 * the split of split3 / the permute kernel */
						const long long K = (long long)p.oh * AT_D, r = orow / K;
						uint16_t *dp = (uint16_t *)p.out + r * 2 * K + (orow - r * K) + d0;
						uint32_t hi[2], lo[2];
						split_bf16x2(x0, x1, hi[0], lo[0]);
						split_bf16x2(x2, x3, hi[1], lo[1]);
						*(uint2 *)dp = make_uint2(hi[0], hi[1]);
						*(uint2 *)(dp + K) = make_uint2(lo[0], lo[1]);
					} else if (p.ofmt == 2) {
						/* f16, flagged as the permute kernel flags it: a
						 * value past 2^15, or four nonzero values all
						 * below 2^-10 */
						const float ax = __builtin_fabsf(x0), ay = __builtin_fabsf(x1);
						const float az = __builtin_fabsf(x2), aw = __builtin_fabsf(x3);
						const float mx = fmaxf(fmaxf(ax, ay), fmaxf(az, aw));
						const bool big = (ax >= 32768.0f && ax <= 3.402823466e38f) ||
								 (ay >= 32768.0f && ay <= 3.402823466e38f) ||
								 (az >= 32768.0f && az <= 3.402823466e38f) ||
								 (aw >= 32768.0f && aw <= 3.402823466e38f);
						if (p.ovf && (big || (mx > 0.0f && mx < 0x1p-10f)))
							*p.ovf = p.ovf_tag;
						*(uint2 *)((uint16_t *)p.out + orow + d0) =
							make_uint2(pack_f16x2(x0, x1), pack_f16x2(x2, x3));
					} else {
						float *O = (float *)p.out + orow;
						*(float4 *)(O + d0) = make_float4(x0, x1, x2, x3);
					}
				} else {
					uint16_t *O = (uint16_t *)p.out + orow;
					*(uint2 *)(O + d0) = make_uint2(at_pack2<DT>(x0, x1), at_pack2<DT>(x2, x3));
				}
			}
	}
}

template <int DT, int NW, bool MASK, bool VD>
__global__ void __launch_bounds__(64 * NW, (at_minb<DT, NW, MASK, VD>())) attn_fwd(AttnArgs p)
{
	using C = AtCfg<DT, NW, VD>;
	static_assert(!VD || !C::SPLIT, "V by direct-to-LDS loads for 16-bit inputs");
	__shared__ __attribute__((aligned(1024))) char smem[C::LDS];
	const int lane = threadIdx.x & 63;
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int h = lane >> 5, l32 = lane & 31;

	/* workgroup -> (head, query block): workgroups are dispatched to the 8
	 * XCDs round-robin, so the nqb blocks of a head are given ids with
	 * one residue mod 8 and run on one XCD, whose L2 then serves the
	 * head's K and V to all of them (the heads past the last whole group
	 * of 8 are laid out plainly) */
	const unsigned L = blockIdx.x, nqb = (unsigned)p.nqb;
	const unsigned g8 = (unsigned)(p.BH / 8) * 8u * nqb;
	unsigned hh, qb;
	if (L < g8) {
		const unsigned sl = L >> 3;
		hh = sl / nqb * 8u + (L & 7u);
		qb = sl % nqb;
	} else {
		hh = (unsigned)(p.BH / 8) * 8u + (L - g8) / nqb;
		qb = (L - g8) % nqb;
	}
	const long long head = hh;
	const int q0w = (int)qb * C::BQ + wave * 32;         /* the wave's first query */
	const int q = q0w + l32;                             /* this lane's query */
	const bool wave_live = q0w < p.Sq;                   /* wave-uniform */
	const bool stager = wave < 4;                        /* threads 0..255 stage K, V */
	const unsigned lds0 = lds_addr_of(smem);
	constexpr int ES = C::SPLIT ? 4 : 2;                 /* input element bytes */

	/* Q^T operand, pre-multiplied by 1/sqrt(64) = 2^-3 (exact): query row
	 * q, d chunk 16c + 8h (hi and lo planes for f32) */
	uint4 qh[4], ql[4];
#pragma unroll
	for (int c = 0; c < 4; ++c) {
		qh[c] = ql[c] = make_uint4(0, 0, 0, 0);
		if (q < p.Sq) {
			if constexpr (C::SPLIT) {
				const float *Q = (const float *)p.q + head * p.hq + (long long)q * AT_D + 16 * c + 8 * h;
				float4 x = *(const float4 *)Q, y = *(const float4 *)(Q + 4);
				x.x *= 0.125f, x.y *= 0.125f, x.z *= 0.125f, x.w *= 0.125f;
				y.x *= 0.125f, y.y *= 0.125f, y.z *= 0.125f, y.w *= 0.125f;
				at_split8(x, y, qh[c], ql[c]);
			} else {
				const uint16_t *Q = (const uint16_t *)p.q + head * p.hq;
				const uint4 r = *(const uint4 *)(Q + (long long)q * AT_D + 16 * c + 8 * h);
				const uint32_t w[4] = {r.x, r.y, r.z, r.w};
				uint32_t o4[4];
#pragma unroll
				for (int i = 0; i < 4; ++i) {
					float lo, hi;
					if constexpr (DT == S3K_F16) {
						lo = f16_to_f32(w[i] & 0xFFFFu), hi = f16_to_f32(w[i] >> 16);
					} else {
						lo = bf16_to_f32(w[i] & 0xFFFFu), hi = bf16_to_f32(w[i] >> 16);
					}
					o4[i] = at_pack2<DT>(lo * 0.125f, hi * 0.125f);
				}
				qh[c] = make_uint4(o4[0], o4[1], o4[2], o4[3]);
			}
		}
	}

	/* the head's K and V as buffers: loads past Sk rows return zeros */
	const unsigned kv_bytes = (unsigned)((long long)p.Sk * AT_D * ES);
	const s3k_i32x4 rk = buf_rsrc(p.k + head * p.hk * ES, kv_bytes);
	const __amdgpu_buffer_rsrc_t bk = __builtin_amdgcn_make_buffer_rsrc(
		(void *)(p.k + head * p.hk * ES), (short)0, (int)kv_bytes, 0x00020000);
	const __amdgpu_buffer_rsrc_t bv = __builtin_amdgcn_make_buffer_rsrc(
		(void *)(p.v + head * p.hk * ES), (short)0, (int)kv_bytes, 0x00020000);
	constexpr unsigned TILE_BYTES = AT_BKV * AT_D * ES;  /* one K or V tile in memory */

	/* 16-bit K tile: 8 KiB = 8 direct-to-LDS instructions of 64 x 16
	 * bytes; wave w issues instructions w, w + NW, ...; slot s of
	 * instruction j holds row s/8, chunk (s%8) ^ swz(row). Rows past Sk
	 * are given an offset past the buffer and read as zeros. */
	unsigned k_off[C::KJ];
#pragma unroll
	for (int t = 0; t < C::KJ; ++t) {
		const int s = (wave + t * NW) * 64 + lane;
		const int row = s / 8, c = (s % 8) ^ lds_swz<8>(row);
		k_off[t] = (unsigned)(row * AT_D * 2 + c * 16);
	}
	auto issue_k = [&](int kt, unsigned slot) {
		const int rows_left = p.Sk - kt * AT_BKV;
#pragma unroll
		for (int t = 0; t < C::KJ; ++t) {
			const int j = wave + t * NW;
			if (j < 8) {
				const int row = (j * 64 + lane) / 8;
				const unsigned o = row < rows_left ? k_off[t] : S3K_OOB;
				dma16s(lds0 + slot + j * 1024, rk, o, (unsigned)kt * TILE_BYTES);
			}
		}
	};

	/* 16-bit V tile (VD): like K, 8 direct-to-LDS instructions, slot s of
	 * instruction j holding key row s/8, chunk (s%8) ^ at_vswz(row) */
	const s3k_i32x4 rv = buf_rsrc(p.v + head * p.hk * ES, kv_bytes);
	unsigned v_off[VD ? C::KJ : 1];
	if constexpr (VD) {
#pragma unroll
		for (int t = 0; t < C::KJ; ++t) {
			const int s = (wave + t * NW) * 64 + lane;
			const int row = s / 8, c = (s % 8) ^ at_vswz(row);
			v_off[t] = (unsigned)(row * AT_D * 2 + c * 16);
		}
	}
	auto issue_v = [&](int kt, unsigned slot) {
		const int rows_left = p.Sk - kt * AT_BKV;
#pragma unroll
		for (int t = 0; t < C::KJ; ++t) {
			const int j = wave + t * NW;
			if (j < 8) {
				const int row = (j * 64 + lane) / 8;
				const unsigned o = row < rows_left ? v_off[t] : S3K_OOB;
				dma16s(lds0 + slot + j * 1024, rv, o, (unsigned)kt * TILE_BYTES);
			}
		}
	};

	/* staging through registers (threads 0..255): f32 K row t/4, d
	 * 16*(t%4)..+15; V keys 4*(t/16)..+3, d 4*(t%16)..+3 */
	const int kr0 = (threadIdx.x & 255) >> 2, kd0 = 16 * (threadIdx.x & 3);
	const int vk0 = 4 * ((threadIdx.x & 255) >> 4), vd0 = 4 * (threadIdx.x & 15);
	const unsigned kst_off = (unsigned)((kr0 * AT_D + kd0) * ES);
	const unsigned vst_off = (unsigned)((vk0 * AT_D + vd0) * ES);
	uint2 vr[4];
	float4 vf[4], kf[4];
	auto load_kv = [&](int kt) {
		const int so = kt * (int)TILE_BYTES;
		if constexpr (C::SPLIT) {
#pragma unroll
			for (int i = 0; i < 4; ++i)
				kf[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
					bk, kst_off + 16 * i, so, 0));
#pragma unroll
			for (int i = 0; i < 4; ++i)
				vf[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
					bv, vst_off + i * AT_D * 4, so, 0));
		} else {
#pragma unroll
			for (int i = 0; i < 4; ++i)
				vr[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(
					bv, vst_off + i * AT_D * 2, so, 0));
		}
	};
	auto store_kv = [&](unsigned kslot, unsigned vslot) {
		char *vt = smem + vslot;
		if constexpr (C::SPLIT) {
			/* K hi/lo planes: logical chunks kd0/8 and kd0/8 + 1 of row kr0 */
			char *st = smem + kslot;
#pragma unroll
			for (int u = 0; u < 2; ++u) {
				uint4 hi, lo;
				at_split8(kf[2 * u], kf[2 * u + 1], hi, lo);
				const int off = (kr0 * 8 + ((kd0 / 8 + u) ^ lds_swz<8>(kr0))) << 4;
				*(uint4 *)(st + off) = hi;
				*(uint4 *)(st + AT_K_BYTES + off) = lo;
			}
			/* V^T hi/lo planes: row d = vd0 + j holds keys vk0..vk0+3 */
			const float e[4][4] = {{vf[0].x, vf[1].x, vf[2].x, vf[3].x},
					       {vf[0].y, vf[1].y, vf[2].y, vf[3].y},
					       {vf[0].z, vf[1].z, vf[2].z, vf[3].z},
					       {vf[0].w, vf[1].w, vf[2].w, vf[3].w}};
#pragma unroll
			for (int j = 0; j < 4; ++j) {
				uint32_t h0, l0, h1, l1;
				at_split2(e[j][0], e[j][1], h0, l0);
				at_split2(e[j][2], e[j][3], h1, l1);
				const int off = (vd0 + j) * AT_VT_PITCH + vk0 * 2;
				*(uint2 *)(vt + off) = make_uint2(h0, h1);
				*(uint2 *)(vt + AT_VT_BYTES + off) = make_uint2(l0, l1);
			}
		} else {
			/* 4x4 transpose of 16-bit values: row j of the result is d vd0+j */
#pragma unroll
			for (int j = 0; j < 4; ++j) {
				const int sh = (j & 1) * 16;
				uint32_t e[4];
#pragma unroll
				for (int i = 0; i < 4; ++i)
					e[i] = ((j < 2 ? vr[i].x : vr[i].y) >> sh) & 0xFFFFu;
				*(uint2 *)(vt + (vd0 + j) * AT_VT_PITCH + vk0 * 2) =
					make_uint2(e[0] | (e[1] << 16), e[2] | (e[3] << 16));
			}
		}
	};

	/* LDS read addresses: K fragment (c, mb) of row 32mb + l32, chunk
	 * (2c + h) ^ swz(row); V^T row 32md + l32 at key 4h */
	unsigned ka[4][2];
#pragma unroll
	for (int c = 0; c < 4; ++c)
#pragma unroll
		for (int mb = 0; mb < 2; ++mb) {
			const int row = 32 * mb + l32;
			ka[c][mb] = lds0 + (unsigned)((row * 8 + ((2 * c + h) ^ lds_swz<8>(row))) << 4);
		}
	const unsigned va = lds0 + (unsigned)(l32 * AT_VT_PITCH + 8 * h);
	/* VD: the V^T operand of O^T += V^T P^T for row d = 32 md + l32 and keys
	 * 16 cc + 4h + {0..3} (lo) / {8..11} (hi) by transposed reads: lane q of
	 * a 16-lane group G addresses key 4 (G >> 1) + q / 4 (+ 8 for hi), d
	 * 32 md + 16 (G & 1) + 4 (q % 4); chunk cc adds 16 rows (2 KiB) */
	unsigned vtr[2][2];
	if constexpr (VD) {
		const int G = lane >> 4, q = lane & 15;
#pragma unroll
		for (int md = 0; md < 2; ++md)
#pragma unroll
			for (int hl = 0; hl < 2; ++hl) {
				const int key = 4 * (G >> 1) + (q >> 2) + 8 * hl;
				const int d = 32 * md + 16 * (G & 1) + 4 * (q & 3);
				vtr[md][hl] = (unsigned)(key * AT_D * 2 +
							 (((d >> 3) ^ at_vswz(key)) << 4) + ((d >> 2) & 1) * 8);
			}
	}

	const float *mrow = MASK ? p.mask + (long long)(q < p.Sq ? q : p.Sq - 1) * p.Sk : nullptr;

	s3k_f32x16 o[2];
#pragma unroll
	for (int md = 0; md < 2; ++md)
#pragma unroll
		for (int r = 0; r < 16; ++r)
			o[md][r] = 0.0f;
	/* running max (base-2 exponent units) and running sum of this lane's
	 * half of the query's keys */
	float m_run = -3.402823466e38f, l_run = 0.0f;
	constexpr float LOG2E = 1.44269504088896341f;
	const int nkt = (p.Sk + AT_BKV - 1) / AT_BKV;

	/* One 64-key tile. P = stage parity (kt & 1), known at compile time so
	 * that every LDS address is a register plus a constant. */
	auto step = [&](auto par, int kt) {
		constexpr int P = decltype(par)::value;
		constexpr unsigned KSLOT = P * C::KS, VSLOT = 2 * C::KS + P * C::VS;
		constexpr unsigned KNEXT = (1 - P) * C::KS, VNEXT = 2 * C::KS + (1 - P) * C::VS;
		const bool more = kt + 1 < nkt;
		/* K(kt) landed and V^T(kt) stored; every wave is past tile kt-1,
		 * whose slots are refilled below */
		wait_vm<0>();
		__syncthreads();
		if (more) {
			if constexpr (!C::SPLIT)
				issue_k(kt + 1, KNEXT);
			if constexpr (VD)
				issue_v(kt + 1, VNEXT);
			else if (stager)
				load_kv(kt + 1);
		}

		if (wave_live) {
			const int kbase = kt * AT_BKV;
			/* mask of this tile: element 4g+e of block mb is key
			 * kbase + 32mb + 8g + 4h + e */
			float4 mk[2][4];
			if constexpr (MASK) {
#pragma unroll
				for (int mb = 0; mb < 2; ++mb)
#pragma unroll
					for (int g = 0; g < 4; ++g) {
						const int key0 = kbase + 32 * mb + 8 * g + 4 * h;
						if (p.mask_vec) {
							mk[mb][g] = key0 < p.Sk ? *(const float4 *)(mrow + key0)
										: make_float4(0.f, 0.f, 0.f, 0.f);
						} else {
							const int last = p.Sk - 1;
							mk[mb][g] = make_float4(mrow[min(key0, last)], mrow[min(key0 + 1, last)],
										mrow[min(key0 + 2, last)], mrow[min(key0 + 3, last)]);
						}
					}
			}

			/* S^T = K Q^T / 8 for keys 32*mb + (row), this lane's query. The
			 * tile is worked in two 32-key halves mb so that the matrix
			 * cores and the VALU overlap inside the wave: scores of half 1
			 * run while the probabilities of half 0 are formed, and P V of
			 * half 0 while those of half 1 are. */
			s3k_f32x16 s[2];
			auto scores_half = [&](int mb) {
#pragma unroll
				for (int r = 0; r < 16; ++r)
					s[mb][r] = 0.0f;
#pragma unroll
				for (int c = 0; c < 4; ++c) {
					const uint4 kh = *(const uint4 *)(smem + (ka[c][mb] - lds0) + KSLOT);
					if constexpr (C::SPLIT) {
						const uint4 kl = *(const uint4 *)(smem + (ka[c][mb] - lds0) + KSLOT + AT_K_BYTES);
						mfma_chunk<C::FAM>(s[mb], kl, qh[c]);
						mfma_chunk<C::FAM>(s[mb], kh, ql[c]);
					}
					mfma_chunk<C::FAM>(s[mb], kh, qh[c]);
				}
			};
			/* mask and keys past Sk (last tile only) for half mb */
			auto finish_half = [&](int mb) {
				if constexpr (MASK) {
#pragma unroll
					for (int g = 0; g < 4; ++g) {
						s[mb][4 * g] += mk[mb][g].x, s[mb][4 * g + 1] += mk[mb][g].y;
						s[mb][4 * g + 2] += mk[mb][g].z, s[mb][4 * g + 3] += mk[mb][g].w;
					}
				}
				if (kbase + AT_BKV > p.Sk) {
#pragma unroll
					for (int r = 0; r < 16; ++r)
						if (kbase + 32 * mb + 8 * (r >> 2) + 4 * h + (r & 3) >= p.Sk)
							s[mb][r] = -__builtin_inff();
				}
			};

			/* probabilities exp2(s*log2(e) - m) of half mb, packed as the
			 * P^T operand of its two 16-key chunks, and their sum */
			uint4 ph[4], pl[4];
			auto probs = [&](int mb) {
				const float nm = -m_run;
				float ts = 0.0f;
#pragma unroll
				for (int sub = 0; sub < 2; ++sub) {
					float pv[8];
#pragma unroll
					for (int e = 0; e < 8; ++e)
						pv[e] = __builtin_amdgcn_exp2f(fmaf(s[mb][8 * sub + e], LOG2E, nm));
					const int cc = 2 * mb + sub;
					if constexpr (C::SPLIT) {
#pragma unroll
						for (int e = 0; e < 8; ++e)
							ts += pv[e];
						at_split8(make_float4(pv[0], pv[1], pv[2], pv[3]),
							  make_float4(pv[4], pv[5], pv[6], pv[7]), ph[cc], pl[cc]);
					} else {
						/* the sum is of the rounded values the MFMA uses */
						ph[cc] = make_uint4(at_pack2<DT>(pv[0], pv[1]), at_pack2<DT>(pv[2], pv[3]),
								    at_pack2<DT>(pv[4], pv[5]), at_pack2<DT>(pv[6], pv[7]));
						ts = at_sum2<DT>(ph[cc].x, ts);
						ts = at_sum2<DT>(ph[cc].y, ts);
						ts = at_sum2<DT>(ph[cc].z, ts);
						ts = at_sum2<DT>(ph[cc].w, ts);
					}
				}
				return ts;
			};
			/* if some lane's sum passed the bound: move the max to the
			 * tile's (at_new_max), rescale what is accumulated, redo half
			 * mb (rare). In settle(0) half 1's scores count as they are
			 * before its mask and range. Without a mask half 1 is finished
			 * after settle(0) (before it the kernel takes 162 registers
			 * instead of 120); with one before it, the raw maximum kept in
			 * raw1 (180 registers instead of 212: 16 x 1369 x 1369 bf16
			 * 79.2 us instead of 83.0). */
			const bool whole = !MASK && kbase + AT_BKV <= p.Sk;
			auto half_max = [&](int mb) {
				float mt = s[mb][0];
#pragma unroll
				for (int r = 1; r < 16; ++r)
					mt = fmaxf(mt, s[mb][r]);
				return mt;
			};
			float raw1 = 0.0f;
			auto settle = [&](int mb, float ts) {
				if (__builtin_amdgcn_ballot_w64(!(ts <= AT_PSUM_MAX))) {
					const float m_new = at_new_max<DT>(m_run, half_max(mb), MASK && !mb ? raw1 : half_max(1 - mb),
									   mb || whole);
					const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
					m_run = m_new;
					l_run *= alpha;
#pragma unroll
					for (int md = 0; md < 2; ++md)
#pragma unroll
						for (int r = 0; r < 16; ++r)
							o[md][r] *= alpha;
					ts = probs(mb);
				}
				l_run += ts;
			};
			/* O^T += V^T P^T over the chunks of half mb: A = V^T rows d,
			 * keys 16cc + 4h + {0..3, 8..11}, as P^T holds them */
			auto pv_half = [&](int mb) {
#pragma unroll
				for (int md = 0; md < 2; ++md) {
					const char *vrow = smem + (va - lds0) + VSLOT + md * 32 * AT_VT_PITCH;
#pragma unroll
					for (int cc = 2 * mb; cc < 2 * mb + 2; ++cc) {
						uint2 lo, hi;
						if constexpr (VD) {
							lo = at_read_tr(smem, VSLOT + cc * 2048 + vtr[md][0]);
							hi = at_read_tr(smem, VSLOT + cc * 2048 + vtr[md][1]);
						} else {
							lo = *(const uint2 *)(vrow + 32 * cc);
							hi = *(const uint2 *)(vrow + 32 * cc + 16);
						}
						const uint4 vh = make_uint4(lo.x, lo.y, hi.x, hi.y);
						if constexpr (C::SPLIT) {
							const uint2 llo = *(const uint2 *)(vrow + AT_VT_BYTES + 32 * cc);
							const uint2 lhi = *(const uint2 *)(vrow + AT_VT_BYTES + 32 * cc + 16);
							mfma_chunk<C::FAM>(o[md], make_uint4(llo.x, llo.y, lhi.x, lhi.y), ph[cc]);
							mfma_chunk<C::FAM>(o[md], vh, pl[cc]);
						}
						mfma_chunk<C::FAM>(o[md], vh, ph[cc]);
					}
				}
			};

			scores_half(0);
			finish_half(0);
			scores_half(1);
			const float ts0 = probs(0);
			if constexpr (MASK) {
				if (__builtin_amdgcn_ballot_w64(!(ts0 <= AT_PSUM_MAX)))
					raw1 = half_max(1);
				finish_half(1);
				settle(0, ts0);
			} else {
				settle(0, ts0);
				finish_half(1);
			}
			pv_half(0);
			const float ts1 = probs(1);
			settle(1, ts1);
			pv_half(1);
		}

		if constexpr (!VD) {
			if (more && stager)
				store_kv(KNEXT, VNEXT);
		}
	};

	/* prologue: tile 0 into slot 0 */
	if constexpr (!C::SPLIT)
		issue_k(0, 0);
	if constexpr (VD) {
		issue_v(0, 2 * C::KS);
	} else if (stager) {
		load_kv(0);
		store_kv(0, 2 * C::KS);
	}
	for (int kt = 0; kt < nkt; kt += 2) {
		step(at_int<0>{}, kt);
		if (kt + 1 < nkt)
			step(at_int<1>{}, kt + 1);
	}

	at_store<DT>(p, o, l_run, head, q, h);
}

/* ------------------------------------------------------------------ */
/* f32 over prepared K and V planes                                     */
/* ------------------------------------------------------------------ */
/* attn_fwd splits each f32 K and V tile into bf16 planes while it stages
 * it, once per block of 128 queries: 81 keys' tiles x 41 query blocks for
 * a head of 5184 tokens, about as many VALU instructions per tile as the
 * softmax needs, 32 staging registers, and tiles that cannot arrive by
 * direct-to-LDS loads. Here the planes are prepared: a K or V row is 256
 * bytes, hi[64] then lo[64] in bf16 (the bytes of the f32 row it replaces),
 * written once by attn_planes_k or by the producer of K and V.
 * The arithmetic per tile is attn_fwd's.
 *   - Loads: K in two LDS slots, V in one (48 KiB, 168 registers: three
 *     workgroups per CU), all by direct-to-LDS loads. At the top of a tile
 *     V of this tile and K of the next are issued; V is waited for, with a
 *     second barrier, when the scores are done.
 *   - KS key groups of four waves work on tiles kt = g mod KS of the same
 *     128 queries and merge through LDS at the end: problems with fewer
 *     query blocks than CUs keep more than one wave per SIMD.
 *   - A mask tile (32 queries x 64 keys per wave) is loaded row by row with
 *     4-byte direct-to-LDS loads (a row of 64 keys is one instruction; any
 *     row pitch), its 16-byte chunks XOR-swizzled by row, one tile ahead:
 *     per-lane loads would touch 32 rows, i.e. 32 cache lines, with each
 *     instruction.
 * Bound by the MFMAs and the softmax's VALU work on the busiest CUs: 16 x
 * 5184 x 5184 319 us, attn_planes_k included, against 382 for attn_fwd
 * (1036 TFLOP/s of bf16 MFMA; counters: MFMA busy 51 %, VALU 40 % of the
 * time, 656 workgroups on 768 places), masked 16 x 1369 51 against 108;
 * 144 heads x 576 over planes that are already stored 44.7 against 55.2
 * (another run, attn_planes_k included: 55.0 against 48.6). Registers
 * matter: the order of finish_half(1) and settle(0) below decides whether
 * the kernel spills at 168 (then 155 us where it takes 105). */
constexpr int AP_TILE = 2 * AT_K_BYTES;              /* hi and lo, 16 KiB */
constexpr int AP_GROUP = 3 * AP_TILE;                /* K, K, V */
constexpr int AP_MASK = 32 * AT_BKV * 4;             /* one wave's mask tile */

/* one dword per lane from global into LDS at lds_addr + 4 * lane */
__device__ __forceinline__ void dma4s(unsigned lds_addr, s3k_i32x4 rsrc, unsigned voff, unsigned soff)
{
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
		     :: "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}

template <int KS, bool MASK>
constexpr int ap_lds()
{
	return KS * (AP_GROUP + (MASK ? 4 * AP_MASK : 0));
}

template <int KS, bool MASK>
__global__ void __launch_bounds__(256 * KS, KS > 1 ? 1 : MASK ? 2 : 3) attn_planes_fwd(AttnArgs p)
{
	__shared__ __attribute__((aligned(1024))) char smem[ap_lds<KS, MASK>()];
	const int lane = threadIdx.x & 63;
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int grp = KS > 1 ? wave >> 2 : 0, w4 = wave & 3;
	const int h = lane >> 5, l32 = lane & 31;

	/* workgroup -> (head, query block) as in attn_fwd */
	const unsigned L = blockIdx.x, nqb = (unsigned)p.nqb;
	const unsigned g8 = (unsigned)(p.BH / 8) * 8u * nqb;
	unsigned hh, qb;
	if (L < g8) {
		const unsigned sl = L >> 3;
		hh = sl / nqb * 8u + (L & 7u);
		qb = sl % nqb;
	} else {
		hh = (unsigned)(p.BH / 8) * 8u + (L - g8) / nqb;
		qb = (L - g8) % nqb;
	}
	const long long head = hh;
	const int q0w = (int)qb * 128 + w4 * 32;
	const int q = q0w + l32;
	const bool wave_live = q0w < p.Sq;
	const unsigned lds0 = lds_addr_of(smem);
	const unsigned kv0 = (unsigned)grp * AP_GROUP; /* this group's K, K, V slots */
	constexpr unsigned V0 = 2 * AP_TILE;
	const unsigned mk0 = (unsigned)(KS * AP_GROUP + wave * AP_MASK);

	uint4 qh[4], ql[4];
#pragma unroll
	for (int c = 0; c < 4; ++c) {
		qh[c] = ql[c] = make_uint4(0, 0, 0, 0);
		if (q < p.Sq) {
			const float *Q = (const float *)p.q + head * p.hq + (long long)q * AT_D + 16 * c + 8 * h;
			float4 x = *(const float4 *)Q, y = *(const float4 *)(Q + 4);
			x.x *= 0.125f, x.y *= 0.125f, x.z *= 0.125f, x.w *= 0.125f;
			y.x *= 0.125f, y.y *= 0.125f, y.z *= 0.125f, y.w *= 0.125f;
			at_split8(x, y, qh[c], ql[c]);
		}
	}

	/* rows past Sk read as zeros (offset past the buffer) */
	const unsigned kv_bytes = (unsigned)((long long)p.Sk * AT_D * 4);
	const s3k_i32x4 rk = buf_rsrc(p.k + head * p.hk * 4, kv_bytes);
	const s3k_i32x4 rv = buf_rsrc(p.v + head * p.hk * 4, kv_bytes);
	constexpr unsigned TILE_BYTES = AT_BKV * AT_D * 4;

	/* a tile is 16 instructions of 1 KiB, four per wave: instruction
	 * w4 + 4t fills rows 8 ((w4 + 4t) % 8).. of plane (w4 + 4t) / 8; slot s
	 * of it holds row s / 8, chunk (s % 8) ^ swizzle(row) */
	unsigned k_off[4], v_off[4];
#pragma unroll
	for (int t = 0; t < 4; ++t) {
		const int j = w4 + 4 * t, s = (j & 7) * 64 + lane, row = s / 8, pl = j >> 3;
		k_off[t] = (unsigned)(row * 256 + pl * 128 + ((s % 8) ^ lds_swz<8>(row)) * 16);
		v_off[t] = (unsigned)(row * 256 + pl * 128 + ((s % 8) ^ at_vswz(row)) * 16);
	}
	auto issue = [&](int kt, unsigned slot, s3k_i32x4 r, const unsigned (&off)[4]) {
		const int rows_left = p.Sk - kt * AT_BKV;
#pragma unroll
		for (int t = 0; t < 4; ++t) {
			const int j = w4 + 4 * t, row = ((j & 7) * 64 + lane) / 8;
			dma16s(lds0 + slot + (unsigned)j * 1024u, r, row < rows_left ? off[t] : S3K_OOB,
			       (unsigned)kt * TILE_BYTES);
		}
	};
	/* mask rows q0w + r, keys of tile kt: LDS row r, slot s holds the
	 * 16-byte chunk s ^ (r & 15). Keys past Sk read the next row (or, past
	 * the mask's end, zeros): their scores become -inf anyway. Rows past Sq
	 * are past the end. */
	const s3k_i32x4 rm = MASK ? buf_rsrc(p.mask, (unsigned)((long long)p.Sq * p.Sk * 4)) : rk;
	auto issue_mask = [&](int kt) {
#pragma unroll
		for (int r = 0; r < 32; ++r) {
			const int row = q0w + r < p.Sq ? q0w + r : p.Sq - 1;
			dma4s(lds0 + mk0 + (unsigned)r * 256u, rm, (unsigned)((lane ^ ((r & 15) << 2)) << 2),
			      (unsigned)(((long long)row * p.Sk + kt * AT_BKV) * 4));
		}
	};

	unsigned ka[4][2];
#pragma unroll
	for (int c = 0; c < 4; ++c)
#pragma unroll
		for (int mb = 0; mb < 2; ++mb) {
			const int row = 32 * mb + l32;
			ka[c][mb] = kv0 + (unsigned)((row * 8 + ((2 * c + h) ^ lds_swz<8>(row))) << 4);
		}
	unsigned vtr[2][2];
	{
		const int G = lane >> 4, q16 = lane & 15;
#pragma unroll
		for (int md = 0; md < 2; ++md)
#pragma unroll
			for (int hl = 0; hl < 2; ++hl) {
				const int key = 4 * (G >> 1) + (q16 >> 2) + 8 * hl;
				const int d = 32 * md + 16 * (G & 1) + 4 * (q16 & 3);
				vtr[md][hl] = kv0 + V0 +
					      (unsigned)(key * AT_D * 2 + (((d >> 3) ^ at_vswz(key)) << 4) +
							 ((d >> 2) & 1) * 8);
			}
	}

	s3k_f32x16 o[2];
#pragma unroll
	for (int md = 0; md < 2; ++md)
#pragma unroll
		for (int r = 0; r < 16; ++r)
			o[md][r] = 0.0f;
	float m_run = -3.402823466e38f, l_run = 0.0f;
	constexpr float LOG2E = 1.44269504088896341f;
	const int nkt = (p.Sk + AT_BKV - 1) / AT_BKV;

	auto step = [&](auto par, int kt) {
		constexpr int P = decltype(par)::value;
		constexpr unsigned KSLOT = P * AP_TILE, KNEXT = (1 - P) * AP_TILE;
		const bool live = KS == 1 || kt < nkt, more = kt + KS < nkt;
		/* K(kt) (and the mask tile) landed; every wave is past its last
		 * reads of the V slot and of the K slot refilled below */
		wait_vm<0>();
		wg_barrier();
		if (live)
			issue(kt, kv0 + V0, rv, v_off);
		if (more)
			issue(kt + KS, kv0 + KNEXT, rk, k_off);

		const int kbase = kt * AT_BKV;
		s3k_f32x16 s[2];
		uint4 ph[4], pl[4];
		float ts0 = 0.0f;
		auto scores_half = [&](int mb) {
#pragma unroll
			for (int r = 0; r < 16; ++r)
				s[mb][r] = 0.0f;
#pragma unroll
			for (int c = 0; c < 4; ++c) {
				const uint4 kh = *(const uint4 *)(smem + ka[c][mb] + KSLOT);
				const uint4 kl = *(const uint4 *)(smem + ka[c][mb] + KSLOT + AT_K_BYTES);
				mfma_chunk<FAM_BF16>(s[mb], kl, qh[c]);
				mfma_chunk<FAM_BF16>(s[mb], kh, ql[c]);
				mfma_chunk<FAM_BF16>(s[mb], kh, qh[c]);
			}
		};
		auto finish_half = [&](int mb) {
			if constexpr (MASK) {
#pragma unroll
				for (int g = 0; g < 4; ++g) {
					const int c = 8 * mb + 2 * g + h; /* chunk of keys 32mb + 8g + 4h.. */
					const float4 m = *(const float4 *)(smem + mk0 + l32 * 256 +
									   ((c ^ (l32 & 15)) << 4));
					s[mb][4 * g] += m.x, s[mb][4 * g + 1] += m.y;
					s[mb][4 * g + 2] += m.z, s[mb][4 * g + 3] += m.w;
				}
			}
			if (kbase + AT_BKV > p.Sk) {
#pragma unroll
				for (int r = 0; r < 16; ++r)
					if (kbase + 32 * mb + 8 * (r >> 2) + 4 * h + (r & 3) >= p.Sk)
						s[mb][r] = -__builtin_inff();
			}
		};
		auto probs = [&](int mb) {
			const float nm = -m_run;
			float ts = 0.0f;
#pragma unroll
			for (int sub = 0; sub < 2; ++sub) {
				float pv[8];
#pragma unroll
				for (int e = 0; e < 8; ++e)
					pv[e] = __builtin_amdgcn_exp2f(fmaf(s[mb][8 * sub + e], LOG2E, nm));
				const int cc = 2 * mb + sub;
#pragma unroll
				for (int e = 0; e < 8; ++e)
					ts += pv[e];
				at_split8(make_float4(pv[0], pv[1], pv[2], pv[3]),
					  make_float4(pv[4], pv[5], pv[6], pv[7]), ph[cc], pl[cc]);
			}
			return ts;
		};
		/* as attn_fwd. One group takes attn_fwd's maxima, for its bits:
		 * half 1's in settle(0) from before its mask and range were
		 * applied. More groups, whose sums are merged in another order
		 * anyway, take the finished scores'. */
		const bool whole = !MASK && kbase + AT_BKV <= p.Sk;
		auto half_max = [&](int mb) {
			float mt = s[mb][0];
#pragma unroll
			for (int r = 1; r < 16; ++r)
				mt = fmaxf(mt, s[mb][r]);
			return mt;
		};
		float raw1 = 0.0f;
		auto settle = [&](int mb, float ts) {
			if (__builtin_amdgcn_ballot_w64(!(ts <= AT_PSUM_MAX))) {
				const float m_new = at_new_max<S3K_F32>(m_run, half_max(mb),
									KS > 1 || mb ? half_max(1 - mb) : raw1,
									KS > 1 || mb || whole);
				const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
				m_run = m_new;
				l_run *= alpha;
#pragma unroll
				for (int md = 0; md < 2; ++md)
#pragma unroll
					for (int r = 0; r < 16; ++r)
						o[md][r] *= alpha;
				ts = probs(mb);
			}
			l_run += ts;
		};
		auto pv_half = [&](int mb) {
#pragma unroll
			for (int md = 0; md < 2; ++md)
#pragma unroll
				for (int cc = 2 * mb; cc < 2 * mb + 2; ++cc) {
					const uint2 hlo = at_read_tr(smem, vtr[md][0] + cc * 2048);
					const uint2 hhi = at_read_tr(smem, vtr[md][1] + cc * 2048);
					const uint2 llo = at_read_tr(smem, vtr[md][0] + cc * 2048 + AT_K_BYTES);
					const uint2 lhi = at_read_tr(smem, vtr[md][1] + cc * 2048 + AT_K_BYTES);
					const uint4 vh = make_uint4(hlo.x, hlo.y, hhi.x, hhi.y);
					mfma_chunk<FAM_BF16>(o[md], make_uint4(llo.x, llo.y, lhi.x, lhi.y), ph[cc]);
					mfma_chunk<FAM_BF16>(o[md], vh, pl[cc]);
					mfma_chunk<FAM_BF16>(o[md], vh, ph[cc]);
				}
		};
		const bool work = wave_live && live;
		if (work) {
			scores_half(0);
			finish_half(0);
			scores_half(1);
			/* (finish before settle: the other order spills registers) */
			ts0 = probs(0);
			if (KS == 1 && __builtin_amdgcn_ballot_w64(!(ts0 <= AT_PSUM_MAX)))
				raw1 = half_max(1);
			finish_half(1);
			settle(0, ts0);
		}
		/* V(kt) has landed in every wave's part; K(kt + KS) may still be
		 * on its way (issued after V) */
		if (more)
			wait_vm<4>();
		else
			wait_vm<0>();
		wg_barrier();
		if constexpr (MASK) {
			/* this wave has read its mask tile (finish_half(1)) */
			__builtin_amdgcn_s_waitcnt(0xC07F); /* lgkmcnt(0) */
			if (wave_live && more)
				issue_mask(kt + KS);
		}
		if (work) {
			pv_half(0);
			const float ts1 = probs(1);
			settle(1, ts1);
			pv_half(1);
		}
	};

	if (grp < nkt) {
		issue(grp, kv0, rk, k_off);
		if (MASK && wave_live)
			issue_mask(grp);
	}
	/* every wave runs the same number of steps (the barriers are
	 * workgroup-wide); a group without a tile left only meets them */
	const int steps = (nkt + KS - 1) / KS;
	for (int it = 0; it < steps; it += 2) {
		step(at_int<0>{}, it * KS + grp);
		if (it + 1 < steps)
			step(at_int<1>{}, (it + 1) * KS + grp);
	}

	if constexpr (KS > 1) {
		/* merge: the groups g > 0 leave their 34 floats per lane in LDS
		 * ([value][lane], one 8.5 KiB region per wave, from offset 0 over
		 * the groups' K and V slots, which no wave reads past this
		 * barrier), group 0 adds them in order */
		__syncthreads();
		constexpr int REG = 34 * 64 * 4;
		static_assert((KS - 1) * 4 * REG <= KS * AP_GROUP, "merge regions fit");
		if (grp > 0) {
			float *r = (float *)(smem + ((grp - 1) * 4 + w4) * REG) + lane;
			r[0] = m_run;
			r[64] = l_run;
#pragma unroll
			for (int md = 0; md < 2; ++md)
#pragma unroll
				for (int e = 0; e < 16; ++e)
					r[(2 + md * 16 + e) * 64] = o[md][e];
		}
		__syncthreads();
		if (grp > 0)
			return;
#pragma unroll
		for (int g = 1; g < KS; ++g) {
			const float *r = (const float *)(smem + ((g - 1) * 4 + w4) * REG) + lane;
			/* the two halves of a query's lanes keep one max (at_max_pair),
			 * so a group without a finite score has -FLT_MAX, sum 0 */
			const float m1 = r[0], m = fmaxf(m_run, m1);
			const float a0 = __builtin_amdgcn_exp2f(m_run - m), a1 = __builtin_amdgcn_exp2f(m1 - m);
			m_run = m;
			l_run = l_run * a0 + r[64] * a1;
#pragma unroll
			for (int md = 0; md < 2; ++md)
#pragma unroll
				for (int e = 0; e < 16; ++e)
					o[md][e] = o[md][e] * a0 + r[(2 + md * 16 + e) * 64] * a1;
		}
	}
	at_store<S3K_F32>(p, o, l_run, head, q, h);
}

/* K and V rows (f32, 64 values) -> hi[64] | lo[64] bf16 rows of the same
 * size; one thread per 8 values. */
__global__ void __launch_bounds__(256) attn_planes_k(const float *__restrict__ k, const float *__restrict__ v,
						     char *__restrict__ ko, char *__restrict__ vo,
						     long long chunks)
{
	const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
	if (i >= 2 * chunks)
		return;
	const bool isv = i >= chunks;
	const long long c = isv ? i - chunks : i;
	const float4 *src = (const float4 *)(isv ? v : k) + 2 * c;
	uint4 hi, lo;
	at_split8(src[0], src[1], hi, lo);
	char *d = (isv ? vo : ko) + (c >> 3) * 256 + (c & 7) * 16;
	*(uint4 *)d = hi;
	*(uint4 *)(d + 128) = lo;
}

/* ------------------------------------------------------------------ */
/* Any head size: one wave per query row                                */
/* ------------------------------------------------------------------ */
struct AttnGArgs {
	const char *q, *k, *v;
	const float *mask;
	char *out;
	int BH, Sq, Sk, D;
	float scale;
	int oh;                 /* > 0: output head-merged (at_out_row) */
	int ofmt;               /* attn_small: AttnArgs' operand forms */
	unsigned *ovf;
	unsigned ovf_tag;
};

template <int DT>
__device__ __forceinline__ float at_ld(const char *base, long long i)
{
	if constexpr (DT == S3K_F32)
		return ((const float *)base)[i];
	else if constexpr (DT == S3K_BF16)
		return bf16_to_f32(((const uint16_t *)base)[i]);
	else
		return f16_to_f32(((const uint16_t *)base)[i]);
}

template <int DT>
__device__ __forceinline__ void at_st(char *base, long long i, float v)
{
	if constexpr (DT == S3K_F32)
		((float *)base)[i] = v;
	else if constexpr (DT == S3K_BF16)
		((uint16_t *)base)[i] = (uint16_t)f32_to_bf16(v);
	else
		((uint16_t *)base)[i] = (uint16_t)f32_to_f16(v);
}

template <int DT, int NACC>
__global__ void __launch_bounds__(256) attn_generic(AttnGArgs p)
{
	__shared__ float qs[4][NACC * 64];
	__shared__ float ps[4][64];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const long long rows = (long long)p.BH * p.Sq;
	long long row = (long long)blockIdx.x * 4 + wave;
	/* every wave runs the same tiles (the barriers are block-wide); a
	 * wave past the last row recomputes it and stores nothing */
	const bool live = row < rows;
	if (!live)
		row = rows - 1;
	const long long head = row / p.Sq;
	const int qi = (int)(row - head * p.Sq);
	const long long kv0 = head * p.Sk * p.D;
	for (int d = lane; d < p.D; d += 64)
		qs[wave][d] = at_ld<DT>(p.q, row * p.D + d);
	__syncthreads();

	float acc[NACC];
#pragma unroll
	for (int i = 0; i < NACC; ++i)
		acc[i] = 0.0f;
	float m_run = -3.402823466e38f, l_run = 0.0f;
	const float *mrow = p.mask ? p.mask + (long long)qi * p.Sk : nullptr;

	for (int t = 0; t < p.Sk; t += 64) {
		const int key = t + lane;
		float s = -__builtin_inff();
		if (key < p.Sk) {
			const long long ko = kv0 + (long long)key * p.D;
			float dot = 0.0f;
			for (int d = 0; d < p.D; ++d)
				dot = fmaf(qs[wave][d], at_ld<DT>(p.k, ko + d), dot);
			s = dot * p.scale;
			if (mrow)
				s += mrow[key];
		}
		float mt = s;
#pragma unroll
		for (int off = 32; off; off >>= 1)
			mt = fmaxf(mt, __shfl_xor(mt, off));
		const float m_new = fmaxf(m_run, mt);
		const float alpha = expf(m_run - m_new);
		const float pj = expf(s - m_new);
		float ls = pj;
#pragma unroll
		for (int off = 32; off; off >>= 1)
			ls += __shfl_xor(ls, off);
		l_run = l_run * alpha + ls;
		m_run = m_new;
		ps[wave][lane] = pj;
		__syncthreads();
#pragma unroll
		for (int i = 0; i < NACC; ++i)
			acc[i] *= alpha;
		const int nk = min(64, p.Sk - t);
		for (int j = 0; j < nk; ++j) {
			const float w = ps[wave][j];
			const long long vo = kv0 + (long long)(t + j) * p.D;
#pragma unroll
			for (int i = 0; i < NACC; ++i) {
				const int d = lane + 64 * i;
				if (d < p.D)
					acc[i] = fmaf(w, at_ld<DT>(p.v, vo + d), acc[i]);
			}
		}
		__syncthreads();
	}
	if (live) {
		const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
#pragma unroll
		for (int i = 0; i < NACC; ++i) {
			const int d = lane + 64 * i;
			if (d < p.D)
				at_st<DT>(p.out, at_out_row(p.oh, head, p.Sq, qi, p.D) + d, acc[i] * inv);
		}
	}
}

/*
 * Attention over few keys (Sk <= 128, D = 64, f32): the text encoder's
 * shapes (cpu_sdpa.c:49-159 per query row, softmax over all keys), where
 * a launch's time is its latency. One workgroup per 16 queries of a head:
 * every load (K, V, the queries, the mask entries) is issued before the
 * first use, so the kernel waits for memory once; K is stored transposed
 * in LDS so that lane j's key j reads are bank-distinct. Wave w owns
 * queries 4w..4w+3 in both phases, lane l keys l and l + 64 for the
 * scores, then output element l. Arithmetic: dot = fmaf over d in
 * order, s = dot * scale + mask, p = expf(s - max), l = butterfly sum,
 * out = (fmaf over keys in order of p * v) * (1 / l), 0 when every score
 * is -inf; for Sk <= 64 these are the steps (and bits) of attn_generic.
 */
constexpr int AS_QB = 16, AS_MAXK = 128, AS_KTP = AS_MAXK + 4;

__global__ void __launch_bounds__(256) attn_small(AttnGArgs p)
{
	__shared__ __attribute__((aligned(16))) float kt[AT_D][AS_KTP];
	__shared__ __attribute__((aligned(16))) float vs[AS_MAXK][AT_D];
	__shared__ __attribute__((aligned(16))) float qs[AS_QB][AT_D];
	__shared__ __attribute__((aligned(16))) float ps[AS_QB][AS_MAXK];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int nqb = (p.Sq + AS_QB - 1) / AS_QB;
	const long long head = blockIdx.x / nqb;
	const int q0 = (int)(blockIdx.x - head * nqb) * AS_QB;
	const int nq = min(AS_QB, p.Sq - q0);
	const float4 *K4 = (const float4 *)p.k + head * p.Sk * (AT_D / 4);
	const float4 *V4 = (const float4 *)p.v + head * p.Sk * (AT_D / 4);
	const float4 *Q4 = (const float4 *)p.q + (head * p.Sq + q0) * (AT_D / 4);
	const int n4 = p.Sk * (AT_D / 4);

	/* every load first */
	constexpr int NL = AS_MAXK * AT_D / 4 / 256; /* float4 of K (and of V) per thread */
	float4 kr[NL], vr[NL];
#pragma unroll
	for (int i = 0; i < NL; ++i) {
		const int idx = min(i * 256 + tid, n4 - 1); /* in bounds; the extra ones unused */
		kr[i] = K4[idx];
		vr[i] = V4[idx];
	}
	const float4 qr = tid < nq * (AT_D / 4) ? Q4[tid] : make_float4(0.f, 0.f, 0.f, 0.f);
	float mk[4][2];
#pragma unroll
	for (int j = 0; j < 4; ++j)
#pragma unroll
		for (int c = 0; c < 2; ++c) {
			const int q = q0 + 4 * wave + j, key = lane + 64 * c;
			mk[j][c] = p.mask && q < p.Sq && key < p.Sk ? p.mask[(long long)q * p.Sk + key]
								      : 0.0f;
		}
#pragma unroll
	for (int i = 0; i < NL; ++i) {
		const int idx = i * 256 + tid;
		if (idx < n4) {
			const int key = idx >> 4, d0 = (idx & 15) * 4;
			kt[d0][key] = kr[i].x;
			kt[d0 + 1][key] = kr[i].y;
			kt[d0 + 2][key] = kr[i].z;
			kt[d0 + 3][key] = kr[i].w;
			*(float4 *)&vs[key][d0] = vr[i];
		}
	}
	*(float4 *)&qs[tid >> 4][(tid & 15) * 4] = qr;
	__syncthreads();

	/* the wave's queries: nqw of 4 exist (wave-uniform); a wave without
	 * any is done (no barrier follows) */
	const int nqw = min(4, p.Sq - (q0 + 4 * wave));
	if (nqw <= 0)
		return;

	/* scores of this wave's queries against keys lane, lane + 64 (the
	 * second only when Sk > 64) */
	float sc[4][2];
#pragma unroll
	for (int j = 0; j < 4; ++j)
		sc[j][0] = sc[j][1] = 0.0f;
	const bool hi = p.Sk > 64;
	auto dots = [&](auto two) {
		constexpr bool TWO = decltype(two)::value != 0;
#pragma unroll 2
		for (int d = 0; d < AT_D; d += 4) {
			float k0[4], k1[4];
#pragma unroll
			for (int e = 0; e < 4; ++e) {
				k0[e] = kt[d + e][lane];
				k1[e] = TWO ? kt[d + e][lane + 64] : 0.0f;
			}
#pragma unroll
			for (int j = 0; j < 4; ++j) {
				const float4 q4 = *(const float4 *)&qs[4 * wave + j][d];
				const float qv[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
				for (int e = 0; e < 4; ++e) {
					sc[j][0] = fmaf(qv[e], k0[e], sc[j][0]);
					if (TWO)
						sc[j][1] = fmaf(qv[e], k1[e], sc[j][1]);
				}
			}
		}
	};
	if (hi)
		dots(at_int<1>{});
	else
		dots(at_int<0>{});
	float inv[4];
#pragma unroll
	for (int j = 0; j < 4; ++j) {
		float s[2], m = -3.402823466e38f;
#pragma unroll
		for (int c = 0; c < 2; ++c) {
			s[c] = -__builtin_inff();
			if (lane + 64 * c < p.Sk) {
				s[c] = sc[j][c] * p.scale;
				if (p.mask)
					s[c] += mk[j][c];
			}
			m = fmaxf(m, s[c]);
		}
#pragma unroll
		for (int off = 32; off; off >>= 1)
			m = fmaxf(m, __shfl_xor(m, off));
		const float p0 = expf(s[0] - m), p1 = hi ? expf(s[1] - m) : 0.0f;
		float l = hi ? p0 + p1 : p0;
#pragma unroll
		for (int off = 32; off; off >>= 1)
			l += __shfl_xor(l, off);
		inv[j] = l > 0.0f ? 1.0f / l : 0.0f;
		ps[4 * wave + j][lane] = p0;
		ps[4 * wave + j][lane + 64] = p1;
	}
	/* the wave reads back only its own rows of ps: its LDS accesses run
	 * in order, so waiting for its writes is enough */
	__builtin_amdgcn_s_waitcnt(0xC07F); /* lgkmcnt(0) */
	__builtin_amdgcn_wave_barrier();

	/* out[q][lane] over the keys in order */
	float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
	int key = 0;
	for (; key + 4 <= p.Sk; key += 4) {
		float v[4];
#pragma unroll
		for (int e = 0; e < 4; ++e)
			v[e] = vs[key + e][lane];
#pragma unroll
		for (int j = 0; j < 4; ++j) {
			const float4 w4 = *(const float4 *)&ps[4 * wave + j][key];
			acc[j] = fmaf(w4.x, v[0], acc[j]);
			acc[j] = fmaf(w4.y, v[1], acc[j]);
			acc[j] = fmaf(w4.z, v[2], acc[j]);
			acc[j] = fmaf(w4.w, v[3], acc[j]);
		}
	}
	for (; key < p.Sk; ++key) {
		const float v = vs[key][lane];
#pragma unroll
		for (int j = 0; j < 4; ++j)
			acc[j] = fmaf(ps[4 * wave + j][key], v, acc[j]);
	}
#pragma unroll
	for (int j = 0; j < 4; ++j) {
		const int q = q0 + 4 * wave + j;
		const float x = acc[j] * inv[j];
		/* the neighbours of the operand forms' pairs and groups of four */
		const float x1 = __shfl_xor(x, 1);
		if (q >= p.Sq)
			continue;
		const long long orow = at_out_row(p.oh, head, p.Sq, q, AT_D);
		if (p.ofmt == 0) {
			((float *)p.out)[orow + lane] = x;
		} else if (p.ofmt == 1) {
			/* bf16 planes [hi|lo] of the merged row, as attn_fwd */
			if (!(lane & 1)) {
				const long long K = (long long)p.oh * AT_D, r = orow / K;
				uint16_t *dp = (uint16_t *)p.out + r * 2 * K + (orow - r * K) + lane;
				uint32_t hi, lo;
				split_bf16x2(x, x1, hi, lo);
				*(uint32_t *)dp = hi;
				*(uint32_t *)(dp + K) = lo;
			}
		} else {
			/* f16, flagged per four values as attn_fwd flags them */
			const float ax = __builtin_fabsf(x);
			float mx = fmaxf(ax, __shfl_xor(ax, 1));
			mx = fmaxf(mx, __shfl_xor(mx, 2));
			const bool big = ax >= 32768.0f && ax <= 3.402823466e38f;
			if (p.ovf && (big || (!(lane & 3) && mx > 0.0f && mx < 0x1p-10f)))
				*p.ovf = p.ovf_tag;
			if (!(lane & 1))
				*(uint32_t *)((uint16_t *)p.out + orow + lane) = pack_f16x2(x, x1);
		}
	}
}

template <int DT>
static void launch_generic(const AttnGArgs &g, hipStream_t st)
{
	const long long rows = (long long)g.BH * g.Sq;
	const dim3 grid((unsigned)((rows + 3) / 4));
	if (g.D <= 64)
		hipLaunchKernelGGL((attn_generic<DT, 1>), grid, dim3(256), 0, st, g);
	else if (g.D <= 128)
		hipLaunchKernelGGL((attn_generic<DT, 2>), grid, dim3(256), 0, st, g);
	else if (g.D <= 256)
		hipLaunchKernelGGL((attn_generic<DT, 4>), grid, dim3(256), 0, st, g);
	else
		hipLaunchKernelGGL((attn_generic<DT, 8>), grid, dim3(256), 0, st, g);
}

} /* namespace s3k */

using namespace s3k;

static int attn_kind_ok(int kind)
{
	return kind == S3K_F32 || kind == S3K_BF16 || kind == S3K_F16;
}

/* Key groups per workgroup of attn_planes_fwd. Up to one workgroup of 128
 * queries per CU the rest of the CU would stay idle, so that workgroup gets
 * three groups of waves (two with a mask, whose tiles take LDS), if there
 * are enough key tiles to share out; past that, one group and up to three
 * workgroups per CU. 16 heads x 1369 queries x 1369 keys (176 workgroups):
 * 42.2 us with one group, 32.5 with three; masked 63.0 and 46.9 with two;
 * 16 x 5184 x 5184 (656): 318 and 323. The tiles asked for grow with the
 * workgroups: 16 x 576 (80 workgroups, 9 tiles) 23 -> 21 us with the pass
 * that makes the planes, 40 x 576 (200) 24 -> 26. */
static int ap_groups(int BH, int Sq, int Sk, bool mask)
{
	const long long wgs = (long long)BH * ((Sq + 127) / 128), nkt = (Sk + AT_BKV - 1) / AT_BKV;
	const bool few = wgs <= 256 && nkt >= 8 && nkt * 16 >= wgs;
	return !few ? 1 : mask ? 2 : 3;
}

static int launch_planes(AttnArgs p, hipStream_t st)
{
	p.nqb = (p.Sq + 127) / 128;
	const int ks = ap_groups(p.BH, p.Sq, p.Sk, p.mask != nullptr);
	const dim3 grid((unsigned)((long long)p.nqb * p.BH));
#define S3K_AP_GO(KS_, M_) hipLaunchKernelGGL((attn_planes_fwd<KS_, M_>), grid, dim3(256 * KS_), 0, st, p)
	if (p.mask && ks == 2)
		S3K_AP_GO(2, true);
	else if (p.mask)
		S3K_AP_GO(1, true);
	else if (ks == 3)
		S3K_AP_GO(3, false);
	else
		S3K_AP_GO(1, false);
#undef S3K_AP_GO
	return (int)hipGetLastError();
}

/* Which kernel runs the problem: S3K_ATTN_MFMA, S3K_ATTN_GENERIC or 0. */
extern "C" int s3k_attn_path(int kind, const void *q, const void *k, const void *v, void *out,
			     int BH, int Sq, int Sk, int D)
{
	if (!attn_kind_ok(kind) || BH < 0 || Sq < 0 || Sk < 0 || D <= 0)
		return 0;
	const long long es = kind == S3K_F32 ? 4 : 2;
	if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & (uintptr_t)(es - 1))
		return 0;
	if (D == AT_D && BH >= 1 && Sq >= 1 && Sk >= 1 && (long long)BH * ((Sq + 127) / 128) < (1LL << 31) &&
	    !(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15u) &&
	    (long long)Sk * AT_D * es <= 0x7FFFFFF0LL)
		return S3K_ATTN_MFMA;
	if (D <= 512 && (long long)BH * Sq / 4 < 0x7FFFFFFFLL)
		return S3K_ATTN_GENERIC;
	return 0;
}

/* The few-keys kernel's conditions (attn_small). */
static bool attn_small_ok(int kind, const void *q, const void *k, const void *v, void *out,
			  int BH, int Sq, int Sk, int D)
{
	return kind == S3K_F32 && D == AT_D && Sk >= 1 && Sk <= AS_MAXK && BH >= 1 && Sq >= 1 &&
	       (long long)BH * ((Sq + AS_QB - 1) / AS_QB) < (1LL << 31) &&
	       !(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15u);
}

/* The kernel s3k_attn_heads(path, ...) runs for these arguments (0: it
 * refuses them). */
static int attn_heads_pick(int path, int kind, const void *q, const void *k, const void *v,
			   void *out, int BH, int Sq, int Sk, int D, int oh, int ofmt)
{
	const int best = s3k_attn_path(kind, q, k, v, out, BH, Sq, Sk, D);
	const bool small = attn_small_ok(kind, q, k, v, out, BH, Sq, Sk, D);
	const bool small_fmt = oh >= 0 && !(oh > 0 && BH % oh) && ofmt >= 0 && ofmt <= 2 &&
			       !(ofmt && oh <= 0);
	if (path == S3K_ATTN_SMALL)
		return small && small_fmt ? S3K_ATTN_SMALL : 0;
	if (path == 0 && small && small_fmt) {
		/* latency-bound sizes, by measured launch time (16 heads, f32,
		 * in a HIP graph): up to 64 scores per head the one-wave-per-row
		 * kernel (1 / 8 queries and keys: 3.3 / 4.4 us against 6.4 /
		 * 6.2 for attn_fwd), from 65 keys the few-keys kernel (77: 9.7
		 * against 11.0), attn_fwd in between (32: 6.5 against 8.5) */
		if ((long long)Sq * Sk <= 64 && !ofmt)
			return S3K_ATTN_GENERIC;
		if (Sk > 64)
			return S3K_ATTN_SMALL;
	}
	if (!best || (path == S3K_ATTN_MFMA && best != S3K_ATTN_MFMA) ||
	    (path != 0 && path != S3K_ATTN_MFMA && path != S3K_ATTN_GENERIC) || oh < 0 ||
	    (oh > 0 && BH % oh) || ofmt < 0 || ofmt > 2 ||
	    (ofmt && (oh <= 0 || kind != S3K_F32 || best != S3K_ATTN_MFMA || path == S3K_ATTN_GENERIC)))
		return 0;
	return path == 0 ? best : path;
}

extern "C" int s3k_attn_heads_path(int kind, const void *q, const void *k, const void *v,
				   void *out, int BH, int Sq, int Sk, int D, int oh, int ofmt)
{
	return attn_heads_pick(0, kind, q, k, v, out, BH, Sq, Sk, D, oh, ofmt);
}

/* attn_planes_fwd reads the mask through one buffer */
static bool ap_fits(const void *mask, int Sq, int Sk)
{
	return !mask || (long long)Sq * Sk * 4 <= 0x7FFFFFF0LL;
}

extern "C" int s3k_attn_planes_ok(const void *q, const void *k, const void *v, const void *mask,
				  void *out, int BH, int Sq, int Sk, int D, int oh, int ofmt)
{
	return attn_heads_pick(0, S3K_F32, q, k, v, out, BH, Sq, Sk, D, oh, ofmt) == S3K_ATTN_MFMA &&
	       ap_fits(mask, Sq, Sk);
}

/* Whether f32 K and V as they are are worth making planes of first. The
 * pass over them is a launch (about 2 us) and their bytes twice; what it
 * gains depends on how the workgroups of 128 queries fill the 256 CUs, two
 * at a time on attn_fwd (one with a mask), three on attn_planes_fwd (two).
 * Heads x queries x keys, attn_fwd against pass + attn_planes_fwd in us:
 *   - no mask, key groups: the gain grows with the key tiles, the pass with
 *     the heads. 14 x 100 x 500 19.2, 19.1; 28 x 100 x 500 19.2, 21.2; 16 x
 *     700 x 700 25.7, 23.8; 28 x 100 x 700 24.9, 25.9; 50 x 128 x 1500 49.6,
 *     45.4; 90 x 128 x 1500 49.5, 54.7; 16 x 1369 x 1369 47.0, 40.7;
 *   - no mask, one group: a round of workgroups saved (513..768: one
 *     instead of two) or a better filled chip (past 1024), if 17 query
 *     blocks share the pass. 32 x 2300 x 300 (576) 32.5, 29.7; 40 x 2500 x
 *     300 (800) 38.8, 41.5; 100 x 3000 x 300 (2400) 91.6, 86.9; 24 x 3000 x
 *     300 (576) 32.0, 28.6; 16 x 2048 x 700 (256) 26.2, 28.7; 1296 x 576 x
 *     576 (5 blocks a head) 431, 466; 16 x 5184 x 5184 (656) 400, 334;
 *   - mask, two groups: by whole pairs of key tiles. 14 x 100 x 500 24.3,
 *     23.7; 28 x 100 x 500 24.4, 25.9; 64 x 128 x 1024 56.7, 46.2; 200 x 128
 *     x 1024 59.6, 67.8; 16 x 1369 x 1369 120, 51;
 *   - mask, one group: past 256 workgroups attn_fwd needs a second round.
 *     64 x 600 x 400 (320) 46.0, 38.7; 200 x 300 x 300 (600) 52.6, 48.2; 64
 *     x 300 x 300 (192) 18.4, 24.7; 200 x 200 x 64 (400) 14.1, 14.5;
 *   - mask rows that attn_fwd cannot load 16 bytes at a time: also below
 *     that. 64 x 300 x 301 27.1, 24.7; 100 x 200 x 301 27.1, 27.6. */
extern "C" size_t s3k_attn_planes_want(int path, int kind, const void *q, const void *k,
				       const void *v, const void *mask, void *out, int BH, int Sq,
				       int Sk, int D, int oh, int ofmt)
{
	const int use = s3h_settings()->attn_planes;
	if (kind != S3K_F32 || use == 0 || (path != 0 && path != S3K_ATTN_MFMA) ||
	    attn_heads_pick(path, kind, q, k, v, out, BH, Sq, Sk, D, oh, ofmt) != S3K_ATTN_MFMA ||
	    !ap_fits(mask, Sq, Sk))
		return 0;
	const long long nqb = (Sq + 127) / 128, nkt = (Sk + AT_BKV - 1) / AT_BKV, wgs = BH * nqb;
	const bool groups = ap_groups(BH, Sq, Sk, mask != nullptr) > 1;
	bool gain;
	if (!mask && groups) {
		gain = BH <= 60 && BH <= 4 * (nkt - 5);
	} else if (!mask) {
		gain = nqb >= 17 && wgs > 512 && (wgs <= 768 || wgs > 1024);
	} else {
		const bool vec = Sk % 4 == 0 && !((uintptr_t)mask & 15u);
		const long long pairs = nkt / 2;
		if (groups)
			gain = !vec || pairs * pairs >= BH;
		else if (wgs > 256)
			gain = nqb >= 2 && nqb + nkt > 3;
		else
			gain = !vec && wgs * nkt >= 256 && nkt >= 3 && (nqb >= 3 || nkt >= 7);
	}
	if (use < 0 && !gain)
		return 0;
	return (size_t)BH * (size_t)Sk * AT_D * 4 * 2;
}

/* The planes of K, then those of V, at dst (s3k_attn_planes_want bytes). */
extern "C" int s3k_attn_planes_make(const void *k, const void *v, void *dst, int BH, int Sk,
				    void *stream)
{
	const long long chunks = (long long)BH * Sk * (AT_D / 8);
	const long long wgs = (2 * chunks + 255) / 256;
	if (wgs <= 0 || wgs >= (1LL << 31))
		return (int)hipErrorInvalidValue;
	hipLaunchKernelGGL(attn_planes_k, dim3((unsigned)wgs), dim3(256), 0, (hipStream_t)stream,
			   (const float *)k, (const float *)v, (char *)dst, (char *)dst + chunks * 32,
			   chunks);
	return (int)hipGetLastError();
}

extern "C" int s3k_attn_heads(int path, int kind, const void *q, const void *k, const void *v,
			      const float *mask, void *out, int BH, int Sq, int Sk, int D, int oh,
			      int ofmt, unsigned *ovf, unsigned ovf_tag, int kvp, void *stream)
{
	path = attn_heads_pick(path, kind, q, k, v, out, BH, Sq, Sk, D, oh, ofmt);
	if (!path || (kvp && (path != S3K_ATTN_MFMA || kind != S3K_F32 || !ap_fits(mask, Sq, Sk))))
		return (int)hipErrorInvalidValue;
	if (path == S3K_ATTN_SMALL) {
		AttnGArgs g{};
		g.q = (const char *)q;
		g.k = (const char *)k;
		g.v = (const char *)v;
		g.mask = mask;
		g.out = (char *)out;
		g.BH = BH;
		g.Sq = Sq;
		g.Sk = Sk;
		g.D = D;
		g.oh = oh;
		g.ofmt = ofmt;
		g.ovf = ovf;
		g.ovf_tag = ovf_tag;
		g.scale = 1.0f / sqrtf((float)D);
		const dim3 grid((unsigned)((long long)BH * ((Sq + AS_QB - 1) / AS_QB)));
		hipLaunchKernelGGL(attn_small, grid, dim3(256), 0, (hipStream_t)stream, g);
		return (int)hipGetLastError();
	}
	if ((long long)BH * Sq == 0)
		return (int)hipSuccess;
	const hipStream_t st = (hipStream_t)stream;
	if (path == S3K_ATTN_GENERIC) {
		AttnGArgs g{};
		g.q = (const char *)q;
		g.k = (const char *)k;
		g.v = (const char *)v;
		g.mask = mask;
		g.out = (char *)out;
		g.BH = BH;
		g.Sq = Sq;
		g.Sk = Sk;
		g.D = D;
		g.oh = oh;
		g.scale = 1.0f / sqrtf((float)D);
		if (kind == S3K_F32)
			launch_generic<S3K_F32>(g, st);
		else if (kind == S3K_BF16)
			launch_generic<S3K_BF16>(g, st);
		else
			launch_generic<S3K_F16>(g, st);
		return (int)hipGetLastError();
	}
	AttnArgs p;
	p.q = (const char *)q;
	p.k = (const char *)k;
	p.v = (const char *)v;
	p.mask = mask;
	p.out = (char *)out;
	p.Sq = Sq;
	p.Sk = Sk;
	p.hq = (long long)Sq * D;
	p.hk = (long long)Sk * D;
	p.mask_vec = mask && (Sk & 3) == 0 && ((uintptr_t)mask & 15u) == 0;
	/* waves per workgroup: 4 (128 queries); 6 and 8 for measurements */
	int nw = 4;
	if (kind != S3K_F32) {
		const int env = s3h_settings()->attn_nw;
		if (env == 4 || env == 6 || env == 8)
			nw = env;
	}
	p.BH = BH;
	p.oh = oh;
	p.ofmt = ofmt;
	p.ovf = ovf;
	p.ovf_tag = ovf_tag;
	p.nqb = (Sq + 32 * nw - 1) / (32 * nw);
	const dim3 grid((unsigned)((long long)p.nqb * BH));
	const dim3 block(64 * nw);
#define S3K_ATTN_GO(DT_, NW_, VD_)                                                          \
	do {                                                                                 \
		if (mask)                                                                    \
			hipLaunchKernelGGL((attn_fwd<DT_, NW_, true, VD_>), grid, block, 0, st, p);  \
		else                                                                         \
			hipLaunchKernelGGL((attn_fwd<DT_, NW_, false, VD_>), grid, block, 0, st, p); \
	} while (0)
	const bool vd = s3h_settings()->attn_vdma != 0;
	if (kvp)
		return launch_planes(p, st);
	if (kind == S3K_F32)
		S3K_ATTN_GO(S3K_F32, 4, false);
	else if (kind == S3K_BF16) {
		if (nw == 4 && vd)
			S3K_ATTN_GO(S3K_BF16, 4, true);
		else if (nw == 4)
			S3K_ATTN_GO(S3K_BF16, 4, false);
		else if (nw == 6)
			S3K_ATTN_GO(S3K_BF16, 6, false);
		else
			S3K_ATTN_GO(S3K_BF16, 8, false);
	} else {
		if (nw == 4 && vd)
			S3K_ATTN_GO(S3K_F16, 4, true);
		else if (nw == 4)
			S3K_ATTN_GO(S3K_F16, 4, false);
		else if (nw == 6)
			S3K_ATTN_GO(S3K_F16, 6, false);
		else
			S3K_ATTN_GO(S3K_F16, 8, false);
	}
#undef S3K_ATTN_GO
	return (int)hipGetLastError();
}
