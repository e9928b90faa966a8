#include "/root/repo/xllm_service_amd/csrc/ops/mfma_rows.h"
#include <cstdio>
#include <vector>
using namespace xllm;
__global__ void k(unsigned* o){ unsigned i=blockIdx.x*256+threadIdx.x; if(i>=65536)return; constexpr float s=0x1p-24f; float z=__uint_as_float(i<<16);
  float d=fmaf(__expf(-z),s,s); float r=__builtin_amdgcn_rcpf(d); float a=z*(s*fmaf(fmaf(-fminf(d,3e38f),r,1.0f),r,r)); float b=(z*s)*r; float c=z*(s*r);
  o[i]=pack_bf16(a,b); o[65536+i]=pack_bf16(a,c);}
int main(){unsigned*d;hipMalloc(&d,65536*8);k<<<256,256>>>(d);std::vector<unsigned>h(131072);hipMemcpy(h.data(),d,65536*8,hipMemcpyDeviceToHost);
 int n=0,m=0;for(int i=0;i<65536;i++){unsigned a=h[i]&0xffff,b=h[i]>>16,c=h[65536+i]>>16;bool na=(a&0x7fff)>0x7f80,nb=(b&0x7fff)>0x7f80;if(a!=b&&!(na&&nb)){n++;if(n<20)printf("%04x: %04x %04x\n",i,a,b);}if(a!=c&&!(na&&(c&0x7fff)>0x7f80))m++;}printf("differ %d, %d of 65536\n",n,m);}
