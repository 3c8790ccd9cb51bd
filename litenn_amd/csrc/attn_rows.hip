// Attention of many query rows with Float32 operands on the matrix cores: the prompt's attention under
// LITENN_HIP_MATMUL_PRECISE, the reference layer with its options (src/LiteNN/Layer/FlashAttnExt.h:100-228) and
// the layered decoders' windows in 32 bits.  The row kernels this stands beside read every key once per query row.
//
//   S^T[key, q]  = K[key, :] . Q[q, :]        A = keys (row-major in LDS), B = queries (registers)
//   O^T[d, q]   += V^T[d, key] . P^T[key, q]  A = values, read transposed from LDS, B = weights (registers)
//
// on v_mfma_f32_32x32x16: a query stays in its lane column through both products, so its running maximum and sum
// live beside its outputs, and the weights leave the first product in the registers the second one takes (the
// order of the keys inside a step is chosen to match; ds_read_b64_tr_b16 turns four keys' rows into the value
// operand).  No operand is rounded to 16 bits:
//   * Float16 keys and values are exact; a query (scaled by a power of two per row) and a softmax weight (scaled
//     by 2^14) are two halves each, hi + lo: two products per operand pair.
//   * Float32 keys, values, queries and weights are three bfloat16 values each, which carry their 24 bits; the
//     six products whose terms reach 2^-24 are formed.
// Scores, softmax and sums are Float32 as in the row kernels.
//
// One wavefront fits a SIMD (256 + 88 registers, most of them the queries' two halves and the outputs), so a tile
// is one chain: stage, 16 products, softmax, 16 products.  200 rows on 1000 keys (32 heads of 128 over 8, mask,
// slopes, soft cap and sinks) take 66 us where the row kernel took 1365, of which 21 are the options' arithmetic;
// against 64 bits 3.8e-7, as before.
#include "common.hpp"
#include "layer_device.hpp"
#include "attn_rows.hpp"

#include <cmath>

namespace litenn_hip
{
	namespace
	{
		typedef _Float16 half8 __attribute__((ext_vector_type(8)));
		typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
		typedef short short4v __attribute__((ext_vector_type(4)));
		typedef float floatx16 __attribute__((ext_vector_type(16)));
		typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
		typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

		constexpr int kKeys = 32; // keys of a tile, queries of a wavefront

		// exp(d) for d <= 0 to about two units in the last place: the product with log2 e is carried in two floats
		__device__ __forceinline__ float exp_f32(float d)
		{
			constexpr float kHi = 1.44269502f, kLo = 1.92596299e-8f, kLn2 = 0.693147182f;
			d = d < -126.0f ? -126.0f : d; // (NaN stays)
			const float t = d * kHi;
			const float r = fmaf(d, kLo, fmaf(d, kHi, -t));
			const float e = __builtin_amdgcn_exp2f(t);
			return fmaf(e, r * kLn2, e);
		}

		// How a Float32 operand is taken apart, and which products of the parts are formed
		struct HalfOperands // keys and values as they are
		{
			typedef half8 frag;
			typedef uint16_t stored;
			static constexpr int kStored = 1, kSplit = 2, kProducts = 2; // pieces of a key or value, of a query or weight
			static constexpr int stored_of[2] = { 0, 0 }, split_of[2] = { 0, 1 };
			static constexpr float kWeightScale = 16384.0f;
			static __device__ __forceinline__ void split(float v, int e, frag (&out)[2])
			{
				out[0][e] = static_cast<_Float16>(v);
				out[1][e] = static_cast<_Float16>(v - static_cast<float>(out[0][e]));
			}
			static __device__ __forceinline__ floatx16 multiply(frag a, frag b, floatx16 c)
			{
				return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
			}
		};
		struct FloatOperands
		{
			typedef bf16x8 frag;
			typedef float stored;
			static constexpr int kStored = 3, kSplit = 3, kProducts = 6;
			static constexpr int stored_of[6] = { 0, 0, 1, 1, 0, 2 }, split_of[6] = { 0, 1, 0, 1, 2, 0 };
			static constexpr float kWeightScale = 1.0f;
			static __device__ __forceinline__ void split(float v, int e, frag (&out)[3])
			{
				out[0][e] = static_cast<__bf16>(v);
				const float r1 = v - static_cast<float>(out[0][e]);
				out[1][e] = static_cast<__bf16>(r1);
				out[2][e] = static_cast<__bf16>(r1 - static_cast<float>(out[1][e]));
			}
			static __device__ __forceinline__ floatx16 multiply(frag a, frag b, floatx16 c)
			{
				return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
			}
		};

		// Detail::ComputeALiBiSlope (FlashAttnExt.h:69-96), in double like the reference
		__device__ inline double row_alibi_slope(int head, int heads, double max_bias)
		{
			int head_log2 = 1;
			while ((head_log2 << 1) <= heads)
			{
				head_log2 <<= 1;
			}
			const double m0 = pow(2.0, -max_bias / static_cast<double>(head_log2));
			const double m1 = pow(2.0, -(max_bias / 2.0) / static_cast<double>(head_log2));
			return head < head_log2 ? pow(m0, static_cast<double>(head + 1)) : pow(m1, static_cast<double>(2 * (head - head_log2) + 1));
		}

		// Bytes between staged rows: keys are read 16 bytes per row by consecutive rows (16 rows cover the 64 banks
		// once), values as four rows of 64 bytes (four rows cover them once).
		template <int D>
		constexpr int key_stride() { return 2 * D + 16; }
		template <int D>
		constexpr int value_stride() { return 2 * D + 64; }

		// A workgroup takes 32 QW query rows of one head; its KW groups of QW wavefronts take the key tiles in turn,
		// each group with its own buffers, and merge at the end.
		template <typename O, int D, int QW, int KW>
		__global__ __launch_bounds__(64 * QW * KW) void attn_rows_kernel(const RowsAttn a)
		{
			typedef typename O::frag frag;
			typedef typename O::stored stored;
			constexpr int KS = key_stride<D>(), VS = value_stride<D>();
			constexpr int kKeyBytes = kKeys * KS, kValueBytes = kKeys * VS; // of one piece
			constexpr int kGroupBytes = O::kStored * (kKeyBytes + kValueBytes);
			extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [KW][keys, values]; later the groups' results
			const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int group = wave / QW, qw = wave % QW;
			const int tid = qw * 64 + lane; // within the group
			const int j = lane & 31, h = lane >> 5;
			// heads are dealt to the XCDs in runs, so that the query heads of one key/value head share an L2
			const int head = (a.heads & 7) == 0 ? static_cast<int>(blockIdx.x & 7) * (a.heads >> 3) + static_cast<int>(blockIdx.x >> 3)
			                                    : static_cast<int>(blockIdx.x);
			const int kv_head = head / a.share;
			const int q_first = (static_cast<int>(gridDim.y) - 1 - static_cast<int>(blockIdx.y)) * (32 * QW); // long runs first
			const int keys = a.keys;
			const long long q_at = a.q_at; // key index of query row 0's own position
			const int row = q_first + 32 * qw + j, row_c = min(row, a.rows - 1);
			// keys [lo, hi) a query sees; [first, last) any of the workgroup's
			const auto sees_from = [&](int i) { return static_cast<int>(max(0ll, q_at + i - a.window + 1)); };
			const auto sees_to = [&](int i) { return a.causal ? static_cast<int>(min(static_cast<long long>(keys), q_at + i + 1)) : keys; };
			const int lo = sees_from(row_c), hi = sees_to(row_c);
			const int first = sees_from(q_first), last = sees_to(min(q_first + 32 * QW, a.rows) - 1);
			const int tiles = (last - first + kKeys - 1) / kKeys;
			const int steps = (tiles + KW - 1) / KW;

			const stored* const kb = static_cast<const stored*>(a.k) + kv_head * a.k_head;
			const stored* const vb = static_cast<const stored*>(a.v) + kv_head * a.v_head;
			const auto buffer_row = [&](int key) {
				key += a.ring_first;
				return a.ring > 0 && key >= a.ring ? key - a.ring : key;
			};

			// ---- the wavefront's queries: B operand of the first product, times 2^shift
			frag q[D / 16][O::kSplit];
			float unscale = 1.0f;
			{
				const float* src = a.q + static_cast<size_t>(row_c) * a.ldq + static_cast<size_t>(head) * a.dim;
				float v[D / 16][8];
				float mx = 0.0f;
#pragma unroll
				for (int s = 0; s < D / 16; ++s)
				{
#pragma unroll
					for (int e = 0; e < 8; ++e)
					{
						const int d = 16 * s + 8 * h + e;
						v[s][e] = d < a.dim ? src[d] : 0.0f;
						const float m = fabsf(v[s][e]);
						mx = m <= 3.402823466e38f ? fmaxf(mx, m) : mx;
					}
				}
				int shift = 0;
				if constexpr (O::kSplit == 2)
				{
					mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
					shift = mx > 0.0f ? min(8 - ilogbf(mx), 126) : 0;
					unscale = ldexpf(1.0f, -shift);
				}
#pragma unroll
				for (int s = 0; s < D / 16; ++s)
				{
#pragma unroll
					for (int e = 0; e < 8; ++e)
					{
						O::split(ldexpf(v[s][e], shift), e, q[s]);
					}
				}
			}
			float slope = 1.0f;
			bool apply_slope = false;
			if (a.mask && a.max_bias > 0.0)
			{
				const double sl = row_alibi_slope(head, a.heads, a.max_bias);
				slope = static_cast<float>(sl);
				apply_slope = sl != 1.0;
			}
			const float* const mask_row = a.mask ? a.mask + static_cast<size_t>(row_c) * keys : nullptr;

			// a dot product's score (the causal mask and the window aside)
			const auto score_of = [&](float v, int key) {
				if (a.apply_scale)
				{
					v = __fmul_rn(v, a.scale);
				}
				if (a.softcap != 0.0f)
				{
					// AddTanh as the layer lowers it (Activation.h:34-50): (exp(2x) - 1) / (exp(2x) + 1), NaN beyond exp's range
					const float ex = exp_f32(__fmul_rn(v, 2.0f));
					v = __fmul_rn(__fsub_rn(ex, 1.0f), __builtin_amdgcn_rcpf(__fadd_rn(ex, 1.0f)));
					if (a.apply_cap)
					{
						v = __fmul_rn(v, a.softcap);
					}
				}
				if (mask_row)
				{
					float mv = mask_row[key];
					if (apply_slope)
					{
						mv = __fmul_rn(mv, slope);
					}
					v = __fadd_rn(v, mv);
				}
				return v;
			};

			// ---- staging: a thread moves 8-element pieces of rows
			uint8_t* const k_lds = lds + group * kGroupBytes;
			uint8_t* const v_lds = k_lds + O::kStored * kKeyBytes;
			constexpr int kRowPieces = D / 8, kPieces = kKeys * kRowPieces / (64 * QW);
			static_assert(kPieces * 64 * QW == kKeys * kRowPieces, "pieces per thread");
			constexpr int kWords = sizeof(stored) / 2; // 16-byte words of a piece
			u32x4 kr[kPieces][kWords], vr[kPieces][kWords];
			const auto request = [&](int tile) {
#pragma unroll
				for (int i = 0; i < kPieces; ++i)
				{
					const int c = tid + 64 * QW * i, key = min(first + tile * kKeys + c / kRowPieces, last - 1), d = (c % kRowPieces) * 8;
					const size_t at = buffer_row(key);
#pragma unroll
					for (int w = 0; w < kWords; ++w)
					{
						kr[i][w] = d < a.dim ? *reinterpret_cast<const u32x4*>(kb + at * a.ldk + d + 4 * w) : u32x4{ 0u, 0u, 0u, 0u };
						vr[i][w] = d < a.vdim ? *reinterpret_cast<const u32x4*>(vb + at * a.ldv + d + 4 * w) : u32x4{ 0u, 0u, 0u, 0u };
					}
				}
			};
			const auto store_piece = [&](uint8_t* dst, int piece_bytes, const u32x4 (&w)[kWords]) {
				if constexpr (O::kStored == 1)
				{
					*reinterpret_cast<u32x4*>(dst) = w[0];
				}
				else
				{
					frag f[O::kStored];
#pragma unroll
					for (int e = 0; e < 8; ++e)
					{
						O::split(__uint_as_float(w[e / 4][e % 4]), e, f);
					}
#pragma unroll
					for (int p = 0; p < O::kStored; ++p)
					{
						*reinterpret_cast<frag*>(dst + p * piece_bytes) = f[p];
					}
				}
			};
			const auto deposit = [&]() {
#pragma unroll
				for (int i = 0; i < kPieces; ++i)
				{
					const int c = tid + 64 * QW * i, key = c / kRowPieces, d = (c % kRowPieces) * 8;
					store_piece(k_lds + key * KS + 2 * d, kKeyBytes, kr[i]);
					store_piece(v_lds + key * VS + 2 * d, kValueBytes, vr[i]);
				}
			};
			const auto meet = [&]() {
				if constexpr (QW > 1)
				{
					__syncthreads();
				}
				else
				{
					__builtin_amdgcn_wave_barrier(); // (a wavefront's LDS accesses keep their order)
				}
			};

			floatx16 o[D / 32];
#pragma unroll
			for (int b = 0; b < D / 32; ++b)
			{
				o[b] = floatx16{};
			}
			float run_m = -INFINITY, run_l = 0.0f; // run_l: of this lane's keys
			if (steps > 0)
			{
				request(min(group, tiles - 1));
			}
			for (int step = 0; step < steps; ++step)
			{
				const int tile = step * KW + group;
				const bool live = tile < tiles; // a group without a tile left goes through the motions on the last one
				const int base = first + min(tile, tiles - 1) * kKeys;
				meet(); // the previous tile has been consumed
				deposit();
				request(min(tile + KW, tiles - 1));
				meet();

				floatx16 s = {};
#pragma unroll
				for (int st = 0; st < D / 16; ++st)
				{
#pragma unroll
					for (int p = 0; p < O::kProducts; ++p)
					{
						const frag kf = *reinterpret_cast<const frag*>(k_lds + O::stored_of[p] * kKeyBytes + j * KS + 32 * st + 16 * h);
						s = O::multiply(kf, q[st][O::split_of[p]], s);
					}
				}
				// lane (j, h) holds keys base + 8 (e / 4) + 4 h + e % 4 of query j
				float sc[16];
				float top = -INFINITY;
#pragma unroll
				for (int e = 0; e < 16; ++e)
				{
					const int key = base + 8 * (e / 4) + 4 * h + (e & 3);
					const bool visible = live && key >= lo && key < hi;
					const float v = score_of(s[e] * unscale, visible ? key : lo);
					sc[e] = visible ? v : -INFINITY;
					top = fmaxf(top, sc[e]);
				}
				top = fmaxf(top, __shfl_xor(top, 32, 64));
				const float new_m = fmaxf(run_m, top);
				const float ref_m = new_m == -INFINITY ? 0.0f : new_m; // (no visible key yet: every exponent is -inf)
				const float corr = exp_f32(run_m - ref_m);
				run_m = new_m;
				float sum = 0.0f;
				frag w[2][O::kSplit];
#pragma unroll
				for (int e = 0; e < 16; ++e)
				{
					const float p = exp_f32(sc[e] - ref_m);
					sum += p;
					O::split(p * O::kWeightScale, e & 7, w[e >> 3]);
				}
				run_l = fmaf(run_l, corr, sum);
				if (__builtin_amdgcn_ballot_w64(corr != 1.0f) != 0)
				{
#pragma unroll
					for (int b = 0; b < D / 32; ++b)
					{
						o[b] *= corr;
					}
				}
				// step u: keys 16 u + 4 h + 0..3 and 16 u + 8 + 4 h + 0..3.  Sixteen lanes read four keys' rows of
				// sixteen dimensions, eight bytes each, and get the four keys of one dimension
				const int v_off = ((lane & 15) >> 2) * VS + (lane & 3) * 8 + ((lane >> 4) & 1) * 32;
#pragma unroll
				for (int u = 0; u < 2; ++u)
				{
#pragma unroll
					for (int b = 0; b < D / 32; ++b)
					{
						frag vf[O::kStored];
#pragma unroll
						for (int p = 0; p < O::kStored; ++p)
						{
							typedef __attribute__((address_space(3))) short4v* lds_short4;
							const uint8_t* at = v_lds + p * kValueBytes + (16 * u + 4 * h) * VS + 64 * b + v_off;
							const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4)(at)));
							const u32x2 y = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4)(at + 8 * VS)));
							vf[p] = __builtin_bit_cast(frag, u32x4{ x.x, x.y, y.x, y.y });
						}
#pragma unroll
						for (int p = 0; p < O::kProducts; ++p)
						{
							o[b] = O::multiply(vf[O::stored_of[p]], w[u][O::split_of[p]], o[b]);
						}
					}
				}
			}
			run_l += __shfl_xor(run_l, 32, 64);

			if constexpr (KW > 1)
			{
				// groups 1 .. KW - 1 hand (maximum, sum, outputs) to group 0, which takes them in order
				float* const xch = reinterpret_cast<float*>(lds);
				constexpr int kWaveFloats = (D / 2 + 2) * 64; // of one wavefront: outputs, maximum, sum
				__syncthreads();
				if (group > 0)
				{
					float* dst = xch + ((group - 1) * QW + qw) * kWaveFloats;
#pragma unroll
					for (int b = 0; b < D / 32; ++b)
					{
#pragma unroll
						for (int e = 0; e < 16; e += 4)
						{
							*reinterpret_cast<float4*>(dst + ((b * 16 + e) / 4 * 64 + lane) * 4) = float4{ o[b][e], o[b][e + 1], o[b][e + 2], o[b][e + 3] };
						}
					}
					dst[D / 2 * 64 + lane] = run_m;
					dst[(D / 2 + 1) * 64 + lane] = run_l;
				}
				__syncthreads();
				if (group > 0)
				{
					return;
				}
				for (int other = 0; other < KW - 1; ++other)
				{
					const float* src = xch + (other * QW + qw) * kWaveFloats;
					const float other_m = src[D / 2 * 64 + lane], other_l = src[(D / 2 + 1) * 64 + lane];
					const float all_m = fmaxf(run_m, other_m), ref_m = all_m == -INFINITY ? 0.0f : all_m;
					const float w0 = exp_f32(run_m - ref_m), w1 = exp_f32(other_m - ref_m);
					run_m = all_m;
					run_l = run_l * w0 + other_l * w1;
#pragma unroll
					for (int b = 0; b < D / 32; ++b)
					{
#pragma unroll
						for (int e = 0; e < 16; e += 4)
						{
							const float4 t = *reinterpret_cast<const float4*>(src + ((b * 16 + e) / 4 * 64 + lane) * 4);
							o[b][e] = o[b][e] * w0 + t.x * w1;
							o[b][e + 1] = o[b][e + 1] * w0 + t.y * w1;
							o[b][e + 2] = o[b][e + 2] * w0 + t.z * w1;
							o[b][e + 3] = o[b][e + 3] * w0 + t.w * w1;
						}
					}
				}
			}
			if (row >= a.rows)
			{
				return;
			}
			// An infinity or a NaN reaches every query of a tile through a weight of zero, or comes out of an operand that
			// was taken apart.  A query whose result is not finite is computed again, key by key over its own keys alone,
			// so that it gets what Float32 arithmetic gives it.
			bool finite = fabsf(run_l) <= 3.402823466e38f;
#pragma unroll
			for (int b = 0; b < D / 32; ++b)
			{
#pragma unroll
				for (int e = 0; e < 16; ++e)
				{
					finite = finite && fabsf(o[b][e]) <= 3.402823466e38f;
				}
			}
			if (__builtin_expect(!finite, 0))
			{
				const auto widen = [](stored v) {
					if constexpr (O::kStored == 1)
					{
						return f16_bits_to_f32(v);
					}
					else
					{
						return v;
					}
				};
				const float* src = a.q + static_cast<size_t>(row) * a.ldq + static_cast<size_t>(head) * a.dim;
				run_m = -INFINITY;
				run_l = 0.0f;
#pragma unroll
				for (int b = 0; b < D / 32; ++b)
				{
					o[b] = floatx16{};
				}
				for (int key = lo; key < hi; ++key)
				{
					const stored* kr0 = kb + static_cast<size_t>(buffer_row(key)) * a.ldk;
					const stored* vr0 = vb + static_cast<size_t>(buffer_row(key)) * a.ldv;
					float dot = 0.0f;
					for (int d = 0; d < a.dim; ++d)
					{
						dot = fmaf(src[d], widen(kr0[d]), dot);
					}
					const float v = score_of(dot, key);
					const float new_m = fmaxf(run_m, v), ref_m = new_m == -INFINITY ? 0.0f : new_m;
					const float corr = expf(run_m - ref_m), p = expf(v - ref_m);
					run_m = new_m;
					run_l = fmaf(run_l, corr, p);
#pragma unroll
					for (int b = 0; b < D / 32; ++b)
					{
#pragma unroll
						for (int e = 0; e < 16; ++e)
						{
							const int d = 32 * b + 8 * (e / 4) + 4 * h + (e & 3);
							o[b][e] = fmaf(p * O::kWeightScale, d < a.vdim ? widen(vr0[d]) : 0.0f, o[b][e] * corr);
						}
					}
				}
			}
			float weight = 1.0f, total = run_l;
			if (a.sinks)
			{
				// the sink joins the row maximum and the denominator, not the values (FlashAttnExt.h:184-212)
				const float sink = a.sinks[head];
				const float all_m = fmaxf(run_m, sink);
				weight = exp_f32(run_m - all_m);
				total = run_l * weight + exp_f32(sink - all_m);
			}
			const float inv = weight / total * (a.out_scale / O::kWeightScale);
			float* const out = a.out + static_cast<size_t>(row) * a.ldo + static_cast<size_t>(head) * a.vdim;
			const float* const gate = a.gate ? a.gate + static_cast<size_t>(row) * a.ldg + static_cast<size_t>(head) * a.vdim : nullptr;
#pragma unroll
			for (int b = 0; b < D / 32; ++b)
			{
#pragma unroll
				for (int e = 0; e < 16; e += 4)
				{
					const int d = 32 * b + 2 * e + 4 * h;
					if (d < a.vdim) // (whole groups of eight)
					{
						float4 v = { o[b][e] * inv, o[b][e + 1] * inv, o[b][e + 2] * inv, o[b][e + 3] * inv };
						if (gate)
						{
							v.x *= sigmoid_f32(gate[d]);
							v.y *= sigmoid_f32(gate[d + 1]);
							v.z *= sigmoid_f32(gate[d + 2]);
							v.w *= sigmoid_f32(gate[d + 3]);
						}
						*reinterpret_cast<float4*>(out + d) = v;
					}
				}
			}
		}

		template <typename O, int D, int QW, int KW>
		void launch_form(const RowsAttn& a, hipStream_t s)
		{
			constexpr size_t tiles = static_cast<size_t>(KW) * O::kStored * kKeys * (key_stride<D>() + value_stride<D>());
			constexpr size_t merge = static_cast<size_t>(KW - 1) * QW * (D / 2 + 2) * 64 * sizeof(float);
			constexpr size_t lds = tiles > merge ? tiles : merge;
			static_assert(lds <= 160 * 1024, "LDS");
			allow_dynamic_lds(reinterpret_cast<const void*>(&attn_rows_kernel<O, D, QW, KW>), lds);
			attn_rows_kernel<O, D, QW, KW><<<dim3(a.heads, (a.rows + 32 * QW - 1) / (32 * QW)), dim3(64 * QW * KW), lds, s>>>(a);
		}

		template <int D>
		void launch_dim(const RowsAttn& a, bool f32, hipStream_t s)
		{
			if (f32)
			{
				launch_form<FloatOperands, D, 2, 2>(a, s);
			}
			// Wavefronts that keep to themselves and share out the keys, except where there are few key tiles (us, 32 heads
			// of 128: 200 rows on 1000 keys 45 against 63 with pairs on shared tiles, 220 rows on 128 keys about even, 33 rows on 33 keys 19 against 14)
			else if (a.keys > 4 * kKeys)
			{
				launch_form<HalfOperands, D, 1, 4>(a, s);
			}
			else
			{
				launch_form<HalfOperands, D, 2, 2>(a, s);
			}
		}
	} // namespace

	// Causal attention of m rows at positions past .. past + m - 1 (operands as in launch_attn_decode)
	bool launch_attn_rows_causal(const float* q, const void* kcache, const void* vcache, int cache_dtype, size_t m,
	                             size_t past, size_t n_head, size_t n_kv_head, size_t head_dim, float* out, hipStream_t s)
	{
		if (!attn_rows_pays(m, past + m, cache_dtype == LITENN_F32) || m > 0x3fffffffu || n_head > 65535 || past + m > 0x3fffffffu)
		{
			return false;
		}
		RowsAttn a;
		a.q = q;
		a.ldq = a.ldo = n_head * head_dim;
		a.k = kcache;
		a.v = vcache;
		a.ldk = a.ldv = n_kv_head * head_dim;
		a.k_head = a.v_head = head_dim;
		a.heads = static_cast<int>(n_head);
		a.share = static_cast<int>(n_head / n_kv_head);
		a.dim = a.vdim = static_cast<int>(head_dim);
		a.rows = static_cast<int>(m);
		a.q_at = static_cast<long long>(past);
		a.keys = static_cast<int>(a.q_at) + a.rows;
		a.apply_scale = true;
		a.scale = static_cast<float>(1.0 / sqrt(static_cast<double>(head_dim)));
		a.out = out;
		return launch_attn_rows(a, cache_dtype == LITENN_F32, s);
	}

	bool launch_attn_rows(const RowsAttn& a, bool f32, hipStream_t s)
	{
		const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
		const int piece = f32 ? 4 : 8; // elements of 16 bytes
		if (a.rows <= 0 || a.heads <= 0 || a.dim % 8 != 0 || a.vdim % 8 != 0 || a.dim <= 0 || a.vdim <= 0 || a.dim > 128 || a.vdim > 128 ||
		    a.ldk % piece != 0 || a.ldv % piece != 0 || a.k_head % piece != 0 || a.v_head % piece != 0 || a.ldo % 4 != 0 ||
		    !aligned(a.k) || !aligned(a.v) || !aligned(a.out) || (a.rows + 31) / 32 > 65535)
		{
			return false;
		}
		if (a.dim <= 64 && a.vdim <= 64)
		{
			launch_dim<64>(a, f32, s);
		}
		else
		{
			launch_dim<128>(a, f32, s);
		}
		return true;
	}
} // namespace litenn_hip
