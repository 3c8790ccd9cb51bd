// A tile of a prompt's windowed attention over expanded keys and values on the matrix cores, for the kernels that take such
// tiles alone or beside other work.
#pragma once

#include "layer_device.hpp"

namespace litenn_hip
{
	// the row of the buffer that holds key row r
	__device__ __forceinline__ int window_row(const WindowAttn& a, int r)
	{
		r += a.kv_first;
		return a.kv_ring > 0 && r >= a.kv_ring ? r - a.kv_ring : r;
	}

	// Matrix-core form: a workgroup takes 64 query rows of one head (16 per wavefront) and walks the
	// keys any of them sees in tiles of 64, staged row-major in LDS (values are read transposed).  Both
	// products are formed transposed (keys x queries, value dimensions x queries), so that a query
	// stays in one lane column: the softmax weights leave the first product in the register layout
	// the second one takes, and the running maximum and sum live beside the outputs.  DK and DV are the
	// head sizes rounded up; what lies beyond the true sizes is zero in LDS and in the queries.
	constexpr int kWinQ = 64, kWinKeys = 64;

	// A staged value row is DV halves, its 32-byte columns permuted by the row: sixteen lanes read 32 bytes of four
	// neighbouring rows, 32 lanes of eight, which then cover all banks.
	template <int DV>
	__device__ __forceinline__ int win_value_at(int key, int piece)
	{
		constexpr int kSame = DV < 128 ? 128 / DV : 1, kColumns = DV < 128 ? DV / 16 : 8; // rows that lie side by side on the banks
		return key * DV + ((piece ^ (((key / kSame) & (kColumns - 1)) << 1)) << 3);
	}

	// PARTS = 2: eight wavefronts, two to sixteen queries: both form the scores and the weights of every key, each half of
	// the value dimensions, so that a query's bits are the same whichever of the two forms it takes.  A query tile is a chain of
	// up to 17 key tiles, with one wavefront a SIMD where there are few of them.
	// us for 777 rows of 16 heads of 128, window 1024, 26.1 -> 24.3, 100 rows 10.5 -> 9.2.  (Halves that take the key tiles
	// in turn and meet at the end take 22.2 and 12.0, but round their weights to bfloat16 against maxima of their own: a row's
	// bits hung on how many heads and rows went with it.)  Values turned by the LDS read instead of two bytes at a time on
	// their way in, masks and rescaling only in tiles that need them, queries and gates asked for all at once: 777 rows
	// 34.5 -> 26.1, 2048 rows of 32 heads 102 -> 71.
	// `tile` of 64 queries of head h; win_lds holds window_tile_lds<DK, DV>() bytes, by 256 PARTS threads.
	template <int DK, int DV, int PARTS>
	__device__ __forceinline__ void window_tile_block(const WindowAttn& a, int h, int tile, uint16_t* win_lds)
	{
		constexpr int KS = DK + 8, kThreads = 256 * PARTS, kBlocks = DV / 16 / PARTS; // 16 value dimensions a block
		uint16_t* const k_lds = win_lds;               // [kWinKeys][KS]
		uint16_t* const v_lds = k_lds + kWinKeys * KS; // [kWinKeys][DV], permuted
		const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) & 3;
		const int first_block = PARTS == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8) * kBlocks;
		const int j = lane & 15, g = lane >> 4;
		const int dim = a.shape.dim, vdim = a.shape.vdim;
		const int q_first = tile * kWinQ;
		const int my_q = q_first + 16 * wave + j;
		const int my_row = min(my_q, a.rows - 1);
		const int my_pos = a.q_base + my_row;
		// of the wavefront's queries
		const int wave_q = q_first + 16 * __builtin_amdgcn_readfirstlane(wave);
		const int first_pos = a.q_base + min(wave_q, a.rows - 1), last_pos = a.q_base + min(wave_q + 15, a.rows - 1);
		// key rows (relative to key_base) any query of the tile sees
		const int lo = max(0, a.q_base + q_first - a.shape.window + 1 - a.key_base);
		const int hi = min(a.keys, a.q_base + min(q_first + kWinQ, a.rows) - a.key_base);
		const uint16_t* const keys = static_cast<const uint16_t*>(a.kv) + h / a.shape.share * a.k_head;
		const uint16_t* const values = static_cast<const uint16_t*>(a.kv) + a.v_first + h / a.shape.share * a.v_head;
		const float scale2 = a.shape.scale * kLog2e; // scores in units of log 2

		bf16x8 q_frag[DK / 32];
		{
			const float* q = a.q + static_cast<size_t>(my_row) * a.ldq + static_cast<size_t>(h) * dim;
			if ((dim & 7) == 0) // whole groups of eight: all on their way before the first is looked at
			{
				floatx4 v[DK / 32][2];
#pragma unroll
				for (int st = 0; st < DK / 32; ++st)
				{
					const int d = 32 * st + 8 * g;
					const floatx4_a4* at = reinterpret_cast<const floatx4_a4*>(q + (d < dim ? d : 0));
					v[st][0] = at[0], v[st][1] = at[1];
				}
#pragma unroll
				for (int st = 0; st < DK / 32; ++st)
				{
					const u32x4 w = { pack_bf16(v[st][0].x, v[st][0].y), pack_bf16(v[st][0].z, v[st][0].w),
						              pack_bf16(v[st][1].x, v[st][1].y), pack_bf16(v[st][1].z, v[st][1].w) };
					q_frag[st] = __builtin_bit_cast(bf16x8, 32 * st + 8 * g < dim ? w : u32x4{ 0u, 0u, 0u, 0u });
				}
			}
			else
			{
#pragma unroll
				for (int st = 0; st < DK / 32; ++st)
				{
					uint32_t w[4];
#pragma unroll
					for (int e = 0; e < 4; ++e)
					{
						const int d = 32 * st + 8 * g + 2 * e;
						w[e] = d < dim ? pack_bf16(q[d], d + 1 < dim ? q[d + 1] : 0.0f) : 0u;
					}
					q_frag[st] = __builtin_bit_cast(bf16x8, u32x4{ w[0], w[1], w[2], w[3] });
				}
			}
		}
		floatx4 o[kBlocks];
#pragma unroll
		for (int b = 0; b < kBlocks; ++b)
		{
			o[b] = floatx4{ 0.0f, 0.0f, 0.0f, 0.0f };
		}
		float run_m = -INFINITY, run_l = 0.0f;
		constexpr int KP = DK / 8, VP = DV / 8;              // 16-byte pieces of a row
		constexpr int KN = kWinKeys * KP / kThreads, VN = kWinKeys * VP / kThreads; // pieces a thread stages
		u32x4 kr[KN], vr[VN];
		const auto request = [&](int base) {
#pragma unroll
			for (int i = 0; i < KN; ++i)
			{
				const int c = tid + kThreads * i, key = min(base + c / KP, hi - 1), d = (c % KP) * 8;
				kr[i] = d < dim ? *reinterpret_cast<const u32x4*>(keys + static_cast<size_t>(window_row(a, key)) * a.ldkv + d)
				                : u32x4{ 0u, 0u, 0u, 0u };
			}
#pragma unroll
			for (int i = 0; i < VN; ++i)
			{
				const int c = tid + kThreads * i, key = min(base + c / VP, hi - 1), e = (c % VP) * 8;
				vr[i] = e < vdim ? *reinterpret_cast<const u32x4*>(values + static_cast<size_t>(window_row(a, key)) * a.ldkv + e)
				                 : u32x4{ 0u, 0u, 0u, 0u };
			}
		};
		request(lo);
		for (int base = lo; base < hi; base += kWinKeys)
		{
			__syncthreads(); // the previous tile has been consumed
#pragma unroll
			for (int i = 0; i < KN; ++i)
			{
				const int c = tid + kThreads * i;
				*reinterpret_cast<u32x4*>(&k_lds[(c / KP) * KS + (c % KP) * 8]) = kr[i];
			}
#pragma unroll
			for (int i = 0; i < VN; ++i)
			{
				const int c = tid + kThreads * i;
				*reinterpret_cast<u32x4*>(&v_lds[win_value_at<DV>(c / VP, c % VP)]) = vr[i];
			}
			request(base + kWinKeys);
			__syncthreads();
			// lane (j, g) gets keys base + 16 b + 4 g + 0..3 of query j
			floatx4 s[4];
#pragma unroll
			for (int b = 0; b < 4; ++b)
			{
				s[b] = floatx4{ 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
				for (int st = 0; st < DK / 32; ++st)
				{
					const bf16x8 kf = *reinterpret_cast<const bf16x8*>(&k_lds[(16 * b + j) * KS + 32 * st + 8 * g]);
					s[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, q_frag[st], s[b], 0, 0, 0);
				}
			}
			// the mask where the tile holds a key that one of the wavefront's queries does not see
			const int pos0 = a.key_base + base + 4 * g;
			float sv[4][4];
			if (a.key_base + base + kWinKeys - 1 > first_pos || last_pos - (a.key_base + base) >= a.shape.window)
			{
#pragma unroll
				for (int b = 0; b < 4; ++b)
				{
#pragma unroll
					for (int r = 0; r < 4; ++r)
					{
						const int back = my_pos - (pos0 + 16 * b + r);
						sv[b][r] = back >= 0 && back < a.shape.window ? s[b][r] * scale2 : -INFINITY;
					}
				}
			}
			else
			{
#pragma unroll
				for (int b = 0; b < 4; ++b)
				{
#pragma unroll
					for (int r = 0; r < 4; ++r)
					{
						sv[b][r] = s[b][r] * scale2;
					}
				}
			}
			float top = -INFINITY;
#pragma unroll
			for (int b = 0; b < 4; ++b)
			{
#pragma unroll
				for (int r = 0; r < 4; ++r)
				{
					top = fmaxf(top, sv[b][r]);
				}
			}
			top = fmaxf(top, __shfl_xor(top, 16, 64));
			top = fmaxf(top, __shfl_xor(top, 32, 64));
			// a tile may hold no visible key of this query: exponents then take 0 as the maximum
			const float new_m = fmaxf(run_m, top);
			const float ref_m = new_m == -INFINITY ? 0.0f : new_m;
			const float corr = exp2_f32(run_m - ref_m);
			run_m = new_m;
			float sum = 0.0f;
			bf16x8 p_frag[2];
#pragma unroll
			for (int ks = 0; ks < 2; ++ks)
			{
				float p[8];
#pragma unroll
				for (int r = 0; r < 4; ++r)
				{
					p[r] = exp2_f32(sv[2 * ks][r] - ref_m);
					p[4 + r] = exp2_f32(sv[2 * ks + 1][r] - ref_m);
				}
#pragma unroll
				for (int e = 0; e < 8; ++e)
				{
					sum += p[e];
				}
				p_frag[ks] = __builtin_bit_cast(bf16x8, u32x4{ pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3]),
				                                               pack_bf16(p[4], p[5]), pack_bf16(p[6], p[7]) });
			}
			run_l = fmaf(run_l, corr, sum);
			if (__any(corr != 1.0f)) // (past the first tiles a maximum seldom moves)
			{
#pragma unroll
				for (int b = 0; b < kBlocks; ++b)
				{
					o[b] *= corr;
				}
			}
			// contraction index 8 g + e of step ks stands for key 16 (2 ks) + 4 g + e (e < 4) and key
			// 16 (2 ks + 1) + 4 g + e - 4 (e >= 4)
#pragma unroll
			for (int b = 0; b < kBlocks; ++b)
			{
#pragma unroll
				for (int ks = 0; ks < 2; ++ks)
				{
					// four keys of sixteen dimensions: lane j of sixteen names eight bytes of a row and gets dimension j
					typedef short short4v __attribute__((ext_vector_type(4)));
					typedef __attribute__((address_space(3))) short4v* lds_short4;
					const int key = 32 * ks + 4 * g + (j >> 2), piece = 2 * (first_block + b) + ((j & 3) >> 1), in = (j & 1) * 4;
					const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4)(&v_lds[win_value_at<DV>(key, piece) + in])));
					const uint2 y = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4)(&v_lds[win_value_at<DV>(key + 16, piece) + in])));
					const bf16x8 vf = __builtin_bit_cast(bf16x8, u32x4{ x.x, x.y, y.x, y.y });
					o[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p_frag[ks], o[b], 0, 0, 0);
				}
			}
		}
		run_l += __shfl_xor(run_l, 16, 64);
		run_l += __shfl_xor(run_l, 32, 64);
		if (my_q >= a.rows)
		{
			return;
		}
		float weight = 1.0f, total = run_l;
		if (a.shape.sink)
		{
			const float sink = a.shape.sink[h] * kLog2e;
			const float all_m = fmaxf(run_m, sink);
			weight = exp2_f32(run_m - all_m);
			total = run_l * weight + exp2_f32(sink - all_m);
		}
		const float inv = weight / total * a.out_scale;
		uint16_t* out = static_cast<uint16_t*>(a.out) + static_cast<size_t>(my_q) * a.ldo + static_cast<size_t>(h) * vdim;
		const float* gate = a.gate ? a.gate + static_cast<size_t>(my_q) * a.ldg + static_cast<size_t>(h) * vdim : nullptr;
		floatx4 gates[kBlocks];
		if (gate)
		{
			if ((vdim & 3) == 0) // whole groups of four, all on their way at once
			{
#pragma unroll
				for (int b = 0; b < kBlocks; ++b)
				{
					const int e = 16 * (first_block + b) + 4 * g;
					gates[b] = *reinterpret_cast<const floatx4_a4*>(gate + (e < vdim ? e : 0));
				}
			}
			else
			{
#pragma unroll
				for (int b = 0; b < kBlocks; ++b)
				{
					gates[b] = load_columns(gate, 16 * (first_block + b) + 4 * g, vdim);
				}
			}
		}
#pragma unroll
		for (int b = 0; b < kBlocks; ++b)
		{
			const int e = 16 * (first_block + b) + 4 * g;
			if (e < vdim)
			{
				floatx4 v = o[b] * inv;
				if (gate)
				{
#pragma unroll
					for (int r = 0; r < 4; ++r)
					{
						v[r] *= e + r < vdim ? sigmoid_f32(gates[b][r]) : 0.0f;
					}
				}
				if ((vdim & 3) == 0 && (reinterpret_cast<size_t>(a.out) & 7) == 0)
				{
					*reinterpret_cast<uint2*>(out + e) = make_uint2(pack_bf16(v.x, v.y), pack_bf16(v.z, v.w));
				}
				else
				{
#pragma unroll
					for (int r = 0; r < 4; ++r)
					{
						if (e + r < vdim)
						{
							out[e + r] = to_bf16(v[r]);
						}
					}
				}
			}
		}
	}

	template <int DK, int DV>
	constexpr size_t window_tile_lds()
	{
		return sizeof(uint16_t) * kWinKeys * (DK + 8 + DV);
	}

	// Whether heads start on whole 16-byte pieces and fit the tiles.
	inline bool window_takes_tiles(const WindowAttn& a)
	{
		return !a.f32 && a.k_head % 8 == 0 && a.v_head % 8 == 0 && a.ldkv % 8 == 0 && a.v_first % 8 == 0 &&
		       (a.ldo % 4 == 0 || a.shape.vdim % 4 != 0) && a.shape.dim <= 256 && a.shape.vdim <= 256;
	}

	// Eight wavefronts where a CU has one workgroup at most (us, four against eight, heads of 128: 32 workgroups 10.5 and 9.1,
	// 208 26.1 and 24.2, 256 33.5 and 31.6, 320 24.0 and 24.0, 512 42.9 and 48.9); wider heads have not the registers for two
	// wavefronts a SIMD.
	inline bool window_shares_queries(size_t workgroups) { return workgroups <= 256; }
} // namespace litenn_hip
