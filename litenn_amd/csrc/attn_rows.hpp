// litenn-hip: attention of many query rows with Float32 operands on the matrix cores (attn_rows.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace litenn_hip
{
	// Query row i of head h sees keys max(0, q_at + i - window + 1) .. (causal: q_at + i), below `keys`.  Strides are
	// in elements; key and value heads are shared by `share` query heads.
	struct RowsAttn
	{
		const float* q = nullptr; // [rows, ldq]: heads of `dim`
		size_t ldq = 0;
		const void *k = nullptr, *v = nullptr; // Float16 or Float32
		size_t ldk = 0, ldv = 0, k_head = 0, v_head = 0;
		int ring = 0, ring_first = 0; // ring > 0: key row r lives at (ring_first + r) modulo ring
		int heads = 0, share = 1, dim = 0, vdim = 0, rows = 0, keys = 0;
		long long q_at = 0;
		long long window = 1ll << 62;
		bool causal = true;
		// score = dot [* scale] [softcap: tanh(.) [* softcap]] [+ mask * slope]
		bool apply_scale = false, apply_cap = false;
		float scale = 1.0f, softcap = 0.0f;
		const float* mask = nullptr; // [rows, keys]
		double max_bias = 0.0;
		const float* sinks = nullptr; // [heads]
		const float* gate = nullptr;  // [rows, ldg]: the result times its sigmoid
		size_t ldg = 0;
		float out_scale = 1.0f;
		float* out = nullptr; // [rows, ldo]
		size_t ldo = 0;
	};

	// Whether the tiles pay, by the kernel each entry point has beside them (us of that kernel and of the tiles, 32 heads over 8 unless said).
	//
	// The causal row kernel: Float16 keys of 64, 8 rows on 96 10.7 / 7.3, of 128, 24 on 1000 29 / 21; Float32 keys, 48 on 1000 65 / 53.
	// (Below some 20000 / sqrt(keys) rows of all heads together its 128-wide form is the faster one, 8 on 128 4.9 / 9.8, 30 on 300
	// 14.6 / 15.0: it could have a line of its own there, which is not drawn.)
	inline bool attn_rows_pay_causal(size_t rows, size_t keys, bool f32) { return rows >= (f32 ? 16u : 8u) && keys >= 96; }
	// The row kernel with options and the window's: fetch::rows_options_tiles, rows_window_tiles (fetch_model.hpp).

	// Returns false, launching nothing, for shapes it does not take: head sizes that are no multiple of 8 or above 128,
	// rows that are not whole 16-byte pieces.
	bool launch_attn_rows(const RowsAttn& a, bool f32, hipStream_t s);
	bool launch_attn_rows_causal(const float* q, const void* kcache, const void* vcache, int cache_dtype, size_t m,
	                             size_t past, size_t n_head, size_t n_kv_head, size_t head_dim, float* out, hipStream_t s);
} // namespace litenn_hip
